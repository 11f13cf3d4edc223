// surrogate.hip -- the learned surrogate in front of the tree pricer: an
// ensemble of MLPs (8 -> 256 x 4 -> 1, SiLU) trained on FP64 tree prices,
// with hand-written BF16 MFMA kernels for the three 256x256 layers (forward,
// backward, weight gradients) and FP32 kernels for the input layer, the
// output layer and Adam.  Inference is one fused kernel per batch tile that
// runs every member, forms the ensemble mean and spread, and queues the
// options the surrogate must not price for the FP64 tree, which then runs in
// the same stream on the compacted list.
//
// Matrix-core layout (v_mfma_f32_32x32x16_bf16, one wavefront of 64 lanes):
// lane l holds A[l%32][8(l/32) .. 8(l/32)+7] and B[8(l/32) .. +7][l%32]; the
// 16 accumulators of lane l are D[8(v/4) + 4(l/32) + v%4][l%32], v = 0..15.
// Every GEMM here is C = A B^T; operands in memory are kept in the order in which
// the lanes read them (weight_at, frag_unit), so a wave's operand is one contiguous
// kilobyte.
//
// Training buffers per member (batch rows b, neurons n, inputs k):
//   a_l^T, dz_l^T  BF16 [n][b]  (operands of the weight-gradient GEMMs)
//   dz_1           FP32 [b][n]
//   W_l            BF16 [n][k] and W_l^T [k][n], refreshed by Adam from FP32 masters
#include "hwt_math.h"
#include "hwt_internal.h"
#include "../../include/hwtsurr.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <new>
#include <random>
#include <sstream>
#include <string>
#include <vector>

using namespace hwt;

namespace {

constexpr int NIN = HWT_SURR_INPUTS;
constexpr int HID = HWT_SURR_HIDDEN;
constexpr int NPAR = HWT_SURR_NPARAMS;
constexpr int PSTRIDE = 200192;          // per-member stride of parameter-shaped vectors
constexpr int LAYER_W = HID * HID;        // elements of one 256x256 weight matrix
constexpr int BATCH_STEP = 128;           // the batch is a multiple (DW_SPLIT parts of whole 16-row blocks)
constexpr int SMALL_PARTS = 4;            // partial sums of the small gradients (W1 and the biases)
constexpr int SMALL_N = HID * (NIN + 4);  // ... their parameters
constexpr int DW_SPLIT = 8;               // split of the batch in the weight-gradient GEMMs
constexpr int HEAD_ROWS = 32;             // rows per partial sum of the output layer's gradients
constexpr int INF_ROWS = 128;             // options per inference workgroup
constexpr int ACT_LD = HID + 8;           // LDS row pitch (bf16) of the inference activations
constexpr double RES = HWT_SURR_RESIDUAL_SCALE;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int woff(int l) { return l == 2 ? HWT_SURR_W2 : (l == 3 ? HWT_SURR_W3 : HWT_SURR_W4); }
constexpr int boff(int l) { return l == 2 ? HWT_SURR_B2 : (l == 3 ? HWT_SURR_B3 : HWT_SURR_B4); }

// BF16 with round-to-nearest-even (the hardware conversion, v_cvt_pk_bf16_f32).
__device__ inline uint16_t to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ inline float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// SiLU on the hardware exp2 and reciprocal (v_exp_f32, v_rcp_f32).
__device__ inline float sigmoidf(float z)
{
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
__device__ inline float silu(float z) { return z * sigmoidf(z); }
__device__ inline float dsilu(float z)
{
    const float s = sigmoidf(z);
    return s * (1.0f + z * (1.0f - s));
}

__device__ inline bf16x8 load_frag(const uint16_t *p)
{
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    return __builtin_bit_cast(bf16x8, v);
}

__device__ inline float wave_sum_f(float v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

struct SOpts {
    int32_t n;
    const double *strike, *maturity, *length;
    const uint16_t *tu, *steps;
    const double *a, *sigma;
    const int8_t *type;
};
struct SYield {
    int32_t n;
    const double *rate;
    const int32_t *day;
};

SOpts sopts(const hwt_options_f64 &o)
{
    return SOpts{o.n, o.strike, o.maturity, o.length, o.term_unit, o.term_steps, o.a, o.sigma, o.type};
}

// ------------------------------------------------------------------ inputs
// Network inputs and the closed-form baseline of option i.  Returns false
// when the option lies outside the training box (or its tree has no exercise
// step inside it), in which case only the tree may price it.
//
// Baseline: the Hull-White zero-coupon-bond option formula (Jamshidian 1989)
// on the tree's own dates T = e dt and S = n dt and the tree's discount bonds
// P(T), P(S) (the same interpolation of the same curve), so it satisfies the
// same put-call parity as the tree and the residual is independent of the
// option type:
//   sigma_p = sigma/a (1 - e^{-a(S-T)}) sqrt((1 - e^{-2aT}) / (2a))
//   h = ln(100 P(S) / (X P(T))) / sigma_p + sigma_p / 2
//   call = 100 P(S) N(h) - X P(T) N(h - sigma_p),  put = call - 100 P(S) + X P(T).
// Lattice phase: the tree's bond values at the exercise step are close to
// exp(c0 - B~ x_j) with x_j = j dr, so the strike sits at node coordinate
// u = (c0 - ln X) / (B~ dr); the tree price is piecewise linear in X between
// nodes, and sin/cos(2 pi u) let the network place that pattern.
// B~ = dt (1 - q^m) / (1 - q), q = e^{-a dt}, m = n - e (discrete bond
// sensitivity); c0 = ln(100 P(S)/P(T)) minus the continuous-time convexity
// terms B sigma^2 (1-e^{-aT})^2 / (2a^2) + B^2 sigma^2 (1 - e^{-2aT}) / (4a).
// Whether option i's parameters lie inside the training box.
__device__ bool surr_param_box(const SOpts &o, int i)
{
    const double X = o.strike[i], Tb = o.maturity[i], L = o.length[i], a = o.a[i], sg = o.sigma[i];
    const int tu = o.tu[i], st = o.steps[i], ty = o.type[i];
    return tu == 365 && (st == 12 || st == 36) && X >= 60.0 && X <= 100.0 && L >= 1.0 && L <= 30.0 &&
           Tb - L >= 1.0 && Tb - L <= 10.0 && a >= 0.01 && a <= 0.2 && sg >= 0.005 && sg <= 0.02 &&
           (ty == 0 || ty == 1);
}

// ... and its tree has the exercise step inside (always so for box parameters:
// expiry >= 1 y puts e at 12 or more, bond >= expiry + 1 y puts n above e);
// c receives the tree constants.
__device__ bool surr_in_box(const SOpts &o, int i, OptConst &c)
{
    if (!surr_param_box(o, i)) return false;
    return option_constants(o.strike[i], o.maturity[i], o.length[i], o.tu[i], o.steps[i], o.a[i], o.sigma[i],
                            o.type[i], 1 << 30, c) == ST_OK &&
           c.e >= 1 && c.n > c.e;
}

template <class YieldFn>
__device__ bool surr_inputs(const SOpts &o, int i, float x[NIN], double &base, const YieldFn &yield)
{
    const double X = o.strike[i], a = o.a[i], sg = o.sigma[i];
    const int tu = o.tu[i], st = o.steps[i], ty = o.type[i];
    OptConst c;
    if (!surr_in_box(o, i, c)) return false;
    const double T = c.e * c.dt, S = c.n * c.dt;
    const double PT = exp(-yield(T, tu) * T);
    const double PS = exp(-yield(S, tu) * S);
    const double Bc = (1.0 - exp(-a * (S - T))) / a;
    const double sp = sg * Bc * sqrt((1.0 - exp(-2.0 * a * T)) / (2.0 * a));
    const double h = log(100.0 * PS / (X * PT)) / sp + 0.5 * sp;
    const double r2 = 0.70710678118654752440;
    // N(h) = erfc(-h/sqrt2)/2; the put uses the upper tails directly
    const double call = 100.0 * PS * 0.5 * erfc(-h * r2) - X * PT * 0.5 * erfc(-(h - sp) * r2);
    const double put = X * PT * 0.5 * erfc((h - sp) * r2) - 100.0 * PS * 0.5 * erfc(h * r2);
    base = (ty == 1) ? put : call;
    const double q = exp(-a * c.dt);
    const double Bd = c.dt * (1.0 - pow(q, (double)(c.n - c.e))) / (1.0 - q);
    const double e1 = 1.0 - exp(-a * T);
    const double c0 = log(100.0 * PS / PT) - Bc * sg * sg * e1 * e1 / (2.0 * a * a) -
                      Bc * Bc * sg * sg * (1.0 - exp(-2.0 * a * T)) / (4.0 * a);
    const double u = (c0 - log(X)) / (Bd * c.dr);
    const double ph = 2.0 * (u - floor(u));
    x[0] = (float)((X - 80.0) / 20.0);
    x[1] = (float)((T - 15.5) / 14.5);
    x[2] = (float)((S - T - 5.5) / 4.5);
    x[3] = (float)((st - 24.0) / 12.0);
    x[4] = (float)((a - 0.105) / 0.095);
    x[5] = (float)((sg - 0.0125) / 0.0075);
    x[6] = (float)sinpi(ph);
    x[7] = (float)cospi(ph);
    return true;
}

__global__ void k_train_inputs(SOpts o, SYield y, const double *__restrict__ price, float *__restrict__ X,
                               float *__restrict__ target, int32_t *__restrict__ bad)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= o.n) return;
    float x[NIN];
    double base = 0.0;
    const bool ok = surr_inputs(o, i, x, base,
                                [&](double t, int tu) { return yield_at(t, tu, y.rate, y.day, y.n); });
#pragma unroll
    for (int k = 0; k < NIN; ++k) X[(size_t)i * NIN + k] = ok ? x[k] : 0.0f;
    target[i] = ok ? (float)((price[i] - base) / RES) : 0.0f;
    if (!ok) atomicAdd(bad, 1);
}

// ---------------------------------------------------------------- training
// Gathers `count` rows of every member into the batch buffers (member pitch
// `pitch` rows); each member has its own order.
__global__ void k_gather(const float *__restrict__ X, const float *__restrict__ target, const int32_t *__restrict__ perm,
                         int64_t perm_stride, int64_t offset, int count, int pitch, float *__restrict__ xb,
                         float *__restrict__ tb, int m0)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    const int m = m0 + blockIdx.y;
    if (r >= count) return;
    const int row = perm[(size_t)blockIdx.y * perm_stride + offset + r];
#pragma unroll
    for (int k = 0; k < NIN; ++k) xb[((size_t)m * pitch + r) * NIN + k] = X[(size_t)row * NIN + k];
    tb[(size_t)m * pitch + r] = target[row];
}

struct Net {
    // per member, strides in elements
    float *P;          // FP32 masters [member][PSTRIDE]
    uint16_t *Wb;      // BF16 [member][3][256*256] (layers 2..4), [n][k] in fragment order (weight_at)
    uint16_t *WbT;     // BF16 transposes [member][3][256*256], [k][n], likewise
};

struct Acts {
    int B;                 // rows per member
    float *xb, *tb;        // [m][B][8], [m][B]
    uint16_t *aT;          // [m][3][256][B]  a1..a3 (bf16), in fragment order (frag_unit)
    uint16_t *dzT;         // [m][3][256][B]  dz2..dz4 (bf16), likewise
    float *dz1;            // [m][B][256]
    float *y;              // [m][B] network outputs
    float *gw;             // [m][3][DW_SPLIT][256*256] weight-gradient partials (layers 2..4)
    float *gs;             // [m][SMALL_PARTS][SMALL_N] partial sums of W1, b1, b2, b3, b4
    float *hp;             // [m][B/HEAD_ROWS][257] head partials (dw5, db5)
    double *loss;          // [m] running sum of squared errors
    float *g;              // [m][PSTRIDE] dense gradient
};

__host__ __device__ inline size_t aoff(const Acts &s, int m, int l) { return (((size_t)m * 3 + (l - 1)) * s.B) * HID; }
__host__ __device__ inline size_t dzoff(const Acts &s, int m, int l) { return (((size_t)m * 3 + (l - 2)) * s.B) * HID; }

// Both transposed batch arrays are kept in the order in which the weight-gradient
// GEMM's matrix fragments read them: 16-byte units of eight batch rows of one
// neuron, the 32 neurons of a block side by side, then the other eight rows of a
// block of 16, then the blocks of neurons.  A fragment load is one contiguous
// kilobyte, and so is what a wave stores.
__host__ __device__ inline size_t frag_unit(int n, int r8)  // neuron, batch row / 8
{
    return ((size_t)(r8 >> 1) * (HID / 32) + (n >> 5)) * 64 + (r8 & 1) * 32 + (n & 31);
}
// The weights likewise: element (row, k) of a 256 x 256 operand A[row][k].  (As rows
// a fragment load was 32 pieces: inference of 475,000 rows 1196 us, now 1085.)
__host__ __device__ inline int weight_at(int row, int k)
{
    return (((row >> 5) * (HID / 16) + (k >> 4)) * 64 + ((k >> 3) & 1) * 32 + (row & 31)) * 8 + (k & 7);
}

// Two floats to a packed BF16 pair (a in the low half), round to nearest
// even, as one v_cvt_pk_bf16_f32 (the value-by-value form costs a convert,
// a shift and an or per pair).
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ inline uint32_t pack_bf16x2(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// --- forward and backward of one tile of the batch
// A workgroup (8 waves) takes TILE_ROWS rows of one member through the whole
// network and back: wave w holds neurons [32w, 32w + 32) of every layer for all 64
// rows, D[neuron][row] = W A^T on the matrix cores (A operand: weights from L2 in
// fragment order; B operand: the layer's BF16 tile in LDS).  The FP32
// pre-activations z1..z3 stay in the accumulator layout in registers until the
// backward pass multiplies by their slopes, so of the 800 MB that a layer at a time
// moves per step of 4 x 8192 rows (z, a, dz and a4 out and back, two layouts) only
// what the weight gradients need leaves the chip: a1..a3 and dz2..dz4 (BF16) and dz1,
// 134 MB.  Registers allow one workgroup per CU; a layer's first weights are
// requested before the barrier that its input waits for.  4 x 8192 rows: 62 us,
// where eight kernels took 344.  (115 us while the compiler kept sigmoids and
// addresses from the forward pass and spilled them, z1 was kept too, and each phase
// loaded its own biases.)
constexpr int TILE_ROWS = 64;
constexpr int TILE_LD = HID + 8;   // LDS row pitch (bf16): rows start 16 bytes on in the banks
constexpr int TILE_LDF = HID + 4;  // ... of the FP32 tile

typedef f32x16 Tile[2];  // value v of block rb: neuron n0 + 8 (v/4) + 4 (lane/32) + v%4, row 32 rb + lane%32

// A wave's weights of one layer, TILE_AHEAD of the 16 fragments in flight.
constexpr int TILE_AHEAD = 8;
struct TileWeights {
    bf16x8 w[TILE_AHEAD];
    const uint16_t *p;
    __device__ void start(const uint16_t *W, int n0, int lane)
    {
        p = W + ((size_t)(n0 >> 5) * (HID / 16) * 64 + lane) * 8;
#pragma unroll
        for (int k = 0; k < TILE_AHEAD; ++k) w[k] = load_frag(p + k * 64 * 8);
    }
};

__device__ inline void tile_gemm(TileWeights &w, const uint16_t *in, int lane, Tile &acc)
{
    const uint16_t *b = in + (lane & 31) * TILE_LD + 8 * (lane >> 5);
    acc[0] = acc[1] = f32x16{};
#pragma unroll
    for (int k = 0; k < HID / 16; ++k) {
        const bf16x8 a = w.w[k % TILE_AHEAD];
        const bf16x8 b0 = load_frag(b + 16 * k), b1 = load_frag(b + 32 * TILE_LD + 16 * k);
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b0, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b1, acc[1], 0, 0, 0);
        if (k + TILE_AHEAD < HID / 16) w.w[k % TILE_AHEAD] = load_frag(w.p + (k + TILE_AHEAD) * 64 * 8);
        // reads no further ahead than that: the scheduler would fetch the whole tile
        if (k % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
}

// The tile's values, rounded to BF16, into LDS: four neurons of a row at a time.
template <class F>
__device__ inline void tile_store(uint16_t *out, int n0, int lane, F &&value)
{
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint2 pk = make_uint2(pack_bf16x2(value(rb, 4 * q), value(rb, 4 * q + 1)),
                                        pack_bf16x2(value(rb, 4 * q + 2), value(rb, 4 * q + 3)));
            *reinterpret_cast<uint2 *>(out + (32 * rb + (lane & 31)) * TILE_LD + n0 + 8 * q + 4 * (lane >> 5)) = pk;
        }
}

// A BF16 tile from LDS to its place in a transposed batch array.
__device__ inline void tile_transposed(const uint16_t *in, uint16_t *T, int r0)
{
    const int n = threadIdx.x & (HID - 1);
#pragma unroll
    for (int i = 0; i < TILE_ROWS / 16; ++i) {
        const int j = (threadIdx.x >> 8) + 2 * i;
        uint32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            v[e] = (uint32_t)in[(8 * j + 2 * e) * TILE_LD + n] | ((uint32_t)in[(8 * j + 2 * e + 1) * TILE_LD + n] << 16);
        reinterpret_cast<uint4 *>(T)[frag_unit(n, r0 / 8 + j)] = make_uint4(v[0], v[1], v[2], v[3]);
    }
}

__device__ inline void tile_bias(Tile &z, const float *bias, int n0, int lane)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 b = *reinterpret_cast<const float4 *>(bias + n0 + 8 * q + 4 * (lane >> 5));
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            z[rb][4 * q] += b.x;
            z[rb][4 * q + 1] += b.y;
            z[rb][4 * q + 2] += b.z;
            z[rb][4 * q + 3] += b.w;
        }
    }
}

// What the compiler would keep beside z from the forward pass for the backward one
// (32 sigmoids a layer, the layer-1 addresses) spills; behind this it computes them
// again.
__device__ inline void forget(f32x16 &v) { asm volatile("" : "+v"(v)); }

// Layers:  z1 = W1 x + b1 (FP32), z_l = a_{l-1} W_l^T + b_l, a_l = silu(z_l);
//   head (FP32): y = w5 . a4 + b5, loss = mean (y - t)^2, dy = 2 (y - t) / B,
//   dz4 = dy w5 * silu'(z4), and per 32 rows the partial sums of dw5 = sum dy a4 and
//   db5 = sum dy;
//   dz_{l-1} = (dz_l W_l) * silu'(z_{l-1}).
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_train_tile(Net net, Acts s, int m0,
                                                                                             int Bn)
{
    __shared__ __attribute__((aligned(16))) uint16_t tile[2][TILE_ROWS * TILE_LD];
    __shared__ __attribute__((aligned(16))) float a4[TILE_ROWS * TILE_LDF];
    __shared__ float dys[TILE_ROWS], lossp[TILE_ROWS / HEAD_ROWS * 4];
    // the member's vectors and the tile's inputs, requested together once
    __shared__ __attribute__((aligned(16))) float w1[HID * NIN], bias[4][HID], w5[HID];
    __shared__ __attribute__((aligned(16))) float xs[TILE_ROWS * NIN];
    __shared__ float target[TILE_ROWS];
    const int m = m0 + blockIdx.y;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int r0 = blockIdx.x * TILE_ROWS, n0 = 32 * wave;
    const float *P = net.P + (size_t)m * PSTRIDE;
    const uint16_t *Wb = net.Wb + (size_t)m * 3 * LAYER_W, *WbT = net.WbT + (size_t)m * 3 * LAYER_W;
    auto layer = [](const uint16_t *W, int l) { return W + (size_t)(l - 2) * LAYER_W; };
    TileWeights w;
    Tile z2, z3, z;
    static_assert(TILE_ROWS * NIN == 512 && HID * NIN == 4 * 512 && HID == 256, "one load each");
    {
        const float4 v = reinterpret_cast<const float4 *>(P + HWT_SURR_W1)[t];
        const float x = s.xb[((size_t)m * s.B + r0) * NIN + t];
        const float y = t < TILE_ROWS ? s.tb[(size_t)m * s.B + r0 + t] : 0.0f;
        const float ba = P[(t < HID ? HWT_SURR_B1 : boff(2) - HID) + t], bb = P[(t < HID ? boff(3) : boff(4) - HID) + t];
        const float v5 = t < HID ? P[HWT_SURR_W5 + t] : 0.0f;
        w.start(layer(Wb, 2), n0, lane);
        reinterpret_cast<float4 *>(w1)[t] = v;
        xs[t] = x;
        bias[t >> 8][t & (HID - 1)] = ba;
        bias[2 + (t >> 8)][t & (HID - 1)] = bb;
        if (t < HID) w5[t] = v5;
        if (t < TILE_ROWS) target[t] = y;
    }
    __syncthreads();
    auto layer1 = [&](Tile &z, int lane) {
        float x[2][NIN];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int k = 0; k < NIN; ++k) x[rb][k] = xs[(32 * rb + (lane & 31)) * NIN + k];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int n = n0 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
            z[0][v] = z[1][v] = bias[0][n];
#pragma unroll
            for (int k = 0; k < NIN; ++k) {
                z[0][v] = fmaf(w1[n * NIN + k], x[0][k], z[0][v]);
                z[1][v] = fmaf(w1[n * NIN + k], x[1][k], z[1][v]);
            }
            // no more than four neurons' weights at a time in registers
            if (v % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
    };
    layer1(z, lane);
    tile_store(tile[0], n0, lane, [&](int rb, int v) { return silu(z[rb][v]); });
    __syncthreads();
    tile_gemm(w, tile[0], lane, z2);
    w.start(layer(Wb, 3), n0, lane);
    tile_transposed(tile[0], s.aT + aoff(s, m, 1), r0);
    tile_bias(z2, bias[1], n0, lane);
    tile_store(tile[1], n0, lane, [&](int rb, int v) { return silu(z2[rb][v]); });
    forget(z2[0]);
    forget(z2[1]);
    __syncthreads();
    tile_gemm(w, tile[1], lane, z3);
    w.start(layer(Wb, 4), n0, lane);
    tile_transposed(tile[1], s.aT + aoff(s, m, 2), r0);
    tile_bias(z3, bias[2], n0, lane);
    tile_store(tile[0], n0, lane, [&](int rb, int v) { return silu(z3[rb][v]); });
    forget(z3[0]);
    forget(z3[1]);
    __syncthreads();
    tile_gemm(w, tile[0], lane, z);
    w.start(layer(WbT, 4), n0, lane);
    tile_transposed(tile[0], s.aT + aoff(s, m, 3), r0);
    tile_bias(z, bias[3], n0, lane);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4 *>(a4 + (32 * rb + (lane & 31)) * TILE_LDF + n0 + 8 * q + 4 * (lane >> 5)) =
                make_float4(silu(z[rb][4 * q]), silu(z[rb][4 * q + 1]), silu(z[rb][4 * q + 2]), silu(z[rb][4 * q + 3]));
    forget(z[0]);
    forget(z[1]);
    __syncthreads();
    {
        // four waves per 32 rows, eight rows each
        constexpr int ROWS = HEAD_ROWS / 4;
        const int first = HEAD_ROWS * (wave >> 2) + (wave & 3);
        const float b5 = P[HWT_SURR_B5];
        float p[ROWS], lsum = 0.0f;
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            p[i] = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) p[i] = fmaf(w5[lane + 64 * q], a4[(first + 4 * i) * TILE_LDF + lane + 64 * q], p[i]);
        }
#pragma unroll
        for (int i = 0; i < ROWS; ++i) p[i] = wave_sum_f(p[i]);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int row = first + 4 * i;
            const float yv = p[i] + b5;
            const float err = yv - target[row];
            if (lane == 0) {
                s.y[(size_t)m * s.B + r0 + row] = yv;
                dys[row] = 2.0f * err / (float)Bn;
            }
            lsum += err * err;
        }
        if (lane == 0) lossp[wave] = lsum;
    }
    __syncthreads();
    {
        const int n = t & (HID - 1), half = t >> 8;
        float dw = 0.0f, db = 0.0f;
#pragma unroll 8
        for (int r = 0; r < HEAD_ROWS; ++r) {
            const float dy = dys[HEAD_ROWS * half + r];
            dw = fmaf(dy, a4[(HEAD_ROWS * half + r) * TILE_LDF + n], dw);
            db += dy;
        }
        float *hp = s.hp + ((size_t)m * (s.B / HEAD_ROWS) + 2 * blockIdx.x + half) * (HID + 1);
        hp[n] = dw;
        if (n == 0) {
            const float *lp = lossp + 4 * half;
            hp[HID] = db;
            atomicAdd(&s.loss[m], (double)(lp[0] + lp[1] + lp[2] + lp[3]));
        }
    }
    {
        const float dy[2] = {dys[lane & 31], dys[32 + (lane & 31)]};
        tile_store(tile[1], n0, lane, [&](int rb, int v) {
            return dy[rb] * w5[n0 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4] * dsilu(z[rb][v]);
        });
    }
    __syncthreads();
    tile_gemm(w, tile[1], lane, z);
    w.start(layer(WbT, 3), n0, lane);
    tile_transposed(tile[1], s.dzT + dzoff(s, m, 4), r0);
    tile_store(tile[0], n0, lane, [&](int rb, int v) { return z[rb][v] * dsilu(z3[rb][v]); });
    __syncthreads();
    tile_gemm(w, tile[0], lane, z);
    w.start(layer(WbT, 2), n0, lane);
    tile_transposed(tile[0], s.dzT + dzoff(s, m, 3), r0);
    tile_store(tile[1], n0, lane, [&](int rb, int v) { return z[rb][v] * dsilu(z2[rb][v]); });
    __syncthreads();
    tile_gemm(w, tile[1], lane, z);
    tile_transposed(tile[1], s.dzT + dzoff(s, m, 2), r0);
    int again = lane;
    asm volatile("" : "+v"(again));
    layer1(z2, again);  // rather than kept: 32 registers
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = z[rb][4 * q + k] * dsilu(z2[rb][4 * q + k]);
            *reinterpret_cast<float4 *>(a4 + (32 * rb + (lane & 31)) * TILE_LDF + n0 + 8 * q + 4 * (lane >> 5)) =
                make_float4(v[0], v[1], v[2], v[3]);
        }
    __syncthreads();
    float4 *dz1 = reinterpret_cast<float4 *>(s.dz1 + ((size_t)m * s.B + r0) * HID);
#pragma unroll
    for (int i = 0; i < TILE_ROWS / 8; ++i)
        dz1[(wave + 8 * i) * (HID / 4) + lane] =
            *reinterpret_cast<const float4 *>(a4 + (wave + 8 * i) * TILE_LDF + 4 * lane);
}

// --- weight gradients
// dW_l[n][k] = sum_b dz_l[b][n] a_{l-1}[b][k], one of DW_SPLIT parts of the batch per
// workgroup and 128 x 128 outputs: each wave 64 x 64, four fragments (a contiguous
// kilobyte each) per four matrix instructions, all layers in one launch, with the
// small gradients: 39 us for 4 x 8192 rows (35 without them), where four launches took
// 127.  Bound by memory: 200 MB, of which 100 are the two operands.
constexpr int DW_TILE = 128, DW_AHEAD = 4;
constexpr int DW_BLOCKS = 3 * (HID / DW_TILE) * (HID / DW_TILE) * DW_SPLIT;  // per member
__device__ inline void weight_gradient(const Acts &s, int m, int block, int Bn)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int split = block % DW_SPLIT, rest = block / DW_SPLIT;
    const int l = 2 + rest / 4, row0 = (rest & 1) * DW_TILE + (wave & 1) * 64, col0 = (rest >> 1 & 1) * DW_TILE + (wave >> 1) * 64;
    const int K = Bn / DW_SPLIT;  // a multiple of 16
    const size_t k0 = (size_t)(split * K / 16) * (HID / 32) * 64 * 8;
    const uint16_t *A = s.dzT + dzoff(s, m, l) + k0 + ((size_t)(row0 >> 5) * 64 + lane) * 8;
    const uint16_t *B = s.aT + aoff(s, m, l - 1) + k0 + ((size_t)(col0 >> 5) * 64 + lane) * 8;
    f32x16 acc[2][2] = {};
    struct Step {
        bf16x8 a0, a1, b0, b1;
    };
    const int steps = K / 16;
    auto load = [&](int k) {
        const size_t at = (size_t)min(k, steps - 1) * (HID / 32) * 64 * 8;
        return Step{load_frag(A + at), load_frag(A + at + 64 * 8), load_frag(B + at), load_frag(B + at + 64 * 8)};
    };
    auto product = [&](const Step &f) {
        acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a0, f.b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a0, f.b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a1, f.b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a1, f.b1, acc[1][1], 0, 0, 0);
    };
    // DW_AHEAD steps' fragments in flight
    Step f[DW_AHEAD];
#pragma unroll
    for (int q = 0; q < DW_AHEAD; ++q) f[q] = load(q);
    int k = 0;
    for (; k + DW_AHEAD <= steps; k += DW_AHEAD) {
#pragma unroll
        for (int q = 0; q < DW_AHEAD; ++q) {
            product(f[q]);
            f[q] = load(k + q + DW_AHEAD);
        }
    }
#pragma unroll
    for (int q = 0; q < DW_AHEAD - 1; ++q)
        if (k + q < steps) product(f[q]);
    float *gw = s.gw + (((size_t)m * 3 + (l - 2)) * DW_SPLIT + split) * LAYER_W;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                gw[(size_t)(row0 + 32 * i + 8 * (v / 4) + 4 * (lane >> 5) + v % 4) * HID + col0 + 32 * j + (lane & 31)] =
                    acc[i][j][v];
}

// Gradients of the input layer and of the biases:
//   dW1[n][i] = sum_b dz1[b][n] x[b][i], db1[n] = sum_b dz1[b][n],
//   db_l[n] = sum_b dz_l[b][n] (l = 2..4).
// The rows of each residue of 256 are summed in order, then the residues by halving
// (c and c ^ 32, 16, .. 1 of every 64), then the four 64s (gradient_of).  A workgroup
// takes one of the 64s, a lane one neuron and the eight residues whose rows lie side by
// side, so every load of a wave is one contiguous piece.  (With a lane per residue a
// load was eight pieces of 16 bytes: 52 us for 4 x 8192 rows, these 23 by themselves,
// and 4 of the launch's 39.)
// The last steps of the halving, over a lane's eight residues.
template <class F>
__device__ inline float halve8(F &&v)
{
    const float a = v(0) + v(4), b = v(1) + v(5), c = v(2) + v(6), d = v(3) + v(7);
    return (a + c) + (b + d);
}

// Orders this wave's LDS accesses on either side.
__device__ inline void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// dW1 and db1: 64 neurons and four of the inputs; wave w takes the rows 8 (w + 4 q) on
// of each 256, q = 0, 1.  x is the same for all lanes: from LDS.
constexpr int IN_BLOCKS = (HID / 64) * SMALL_PARTS * 2, IN_AHEAD = 8;
__device__ inline void input_gradient(const Acts &s, int m, int block, int Bn, float *lds)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kh = block & 1, part = block / 2 % SMALL_PARTS, n = block / 2 / SMALL_PARTS * 64 + lane;
    const float *dz1 = s.dz1 + (size_t)m * s.B * HID + n;
    const float *xb = s.xb + (size_t)m * s.B * NIN + 4 * kh;
    float *xw = lds + wave * (4 * 8 * IN_AHEAD);  // the wave's x rows of one round
    float acc[2][8][5] = {};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        // rounds of IN_AHEAD 256s: the loads of all, then their sums
        for (int row = 64 * part + 8 * (wave + 4 * q); row < Bn; row += 256 * IN_AHEAD) {
            const int last = (Bn - 1 - row) / 256;  // of this round's, the last 256 that has the rows
            float d[IN_AHEAD][8];
            const float4 x = *reinterpret_cast<const float4 *>(
                xb + (size_t)(row + 256 * min(lane / 8 % IN_AHEAD, last) + lane % 8) * NIN);
#pragma unroll
            for (int i = 0; i < IN_AHEAD; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) d[i][e] = dz1[(size_t)(row + 256 * min(i, last) + e) * HID];
            if (lane < 8 * IN_AHEAD) *reinterpret_cast<float4 *>(xw + 4 * lane) = x;
            wave_order();
#pragma unroll
            for (int i = 0; i < IN_AHEAD; ++i)
                if (i <= last)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float4 xr = *reinterpret_cast<const float4 *>(xw + 4 * (8 * i + e));
                        acc[q][e][0] = fmaf(d[i][e], xr.x, acc[q][e][0]);
                        acc[q][e][1] = fmaf(d[i][e], xr.y, acc[q][e][1]);
                        acc[q][e][2] = fmaf(d[i][e], xr.z, acc[q][e][2]);
                        acc[q][e][3] = fmaf(d[i][e], xr.w, acc[q][e][3]);
                        acc[q][e][4] += d[i][e];
                    }
            wave_order();
        }
    }
    float v[40];
#pragma unroll
    for (int k = 0; k < 40; ++k) v[k] = acc[0][k / 5][k % 5] + acc[1][k / 5][k % 5];
#pragma unroll
    for (int h = 2; h >= 1; h >>= 1) {  // residues ^ 16, then ^ 8: the other waves
        __syncthreads();
        if (wave >= h && wave < 2 * h)
#pragma unroll
            for (int k = 0; k < 40; ++k) lds[((wave - h) * 40 + k) * 64 + lane] = v[k];
        __syncthreads();
        if (wave < h)
#pragma unroll
            for (int k = 0; k < 40; ++k) v[k] += lds[(wave * 40 + k) * 64 + lane];
    }
    if (wave == 0) {
        float *gs = s.gs + ((size_t)m * SMALL_PARTS + part) * SMALL_N;
#pragma unroll
        for (int k = 0; k < 4; ++k) gs[HWT_SURR_W1 + n * NIN + 4 * kh + k] = halve8([&](int e) { return v[5 * e + k]; });
        if (kh == 0) gs[HWT_SURR_B1 + n] = halve8([&](int e) { return v[5 * e + 4]; });
    }
}

// db_l: 32 neurons of one layer; wave w takes the 16 rows 16 (4 part + w) on of each 256.
constexpr int BIAS_BLOCKS = 3 * (HID / 32) * SMALL_PARTS, BIAS_AHEAD = 8;
__device__ inline void bias_gradient(const Acts &s, int m, int block, int Bn, float *lds)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = block % SMALL_PARTS, nb = block / SMALL_PARTS % (HID / 32), l = 2 + block / SMALL_PARTS / (HID / 32);
    const uint16_t *T = s.dzT + dzoff(s, m, l) + ((size_t)nb * 64 + lane) * 8;
    float acc[8] = {};
    auto load = [&](int r16) { return *reinterpret_cast<const uint4 *>(T + (size_t)r16 * HID * 16); };
    auto add = [&](const uint4 &u) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += __uint_as_float(e & 1 ? w[e / 2] & 0xffff0000u : w[e / 2] << 16);
    };
    int r16 = 4 * part + wave;
    const int end = Bn / 16;
    for (; r16 + 16 * (BIAS_AHEAD - 1) < end; r16 += 16 * BIAS_AHEAD) {
        uint4 u[BIAS_AHEAD];
#pragma unroll
        for (int i = 0; i < BIAS_AHEAD; ++i) u[i] = load(r16 + 16 * i);
#pragma unroll
        for (int i = 0; i < BIAS_AHEAD; ++i) add(u[i]);
    }
    for (; r16 < end; r16 += 16) add(load(r16));
#pragma unroll
    for (int h = 2; h >= 1; h >>= 1) {  // residues ^ 32, then ^ 16: the other waves
        __syncthreads();
        if (wave >= h && wave < 2 * h)
#pragma unroll
            for (int e = 0; e < 8; ++e) lds[((wave - h) * 8 + e) * 64 + lane] = acc[e];
        __syncthreads();
        if (wave < h)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += lds[(wave * 8 + e) * 64 + lane];
    }
    if (wave == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], 32, 64);
        if (lane < 32)
            s.gs[((size_t)m * SMALL_PARTS + part) * SMALL_N + HWT_SURR_B1 + (l - 1) * HID + 32 * nb + lane] =
                halve8([&](int e) { return acc[e]; });
    }
}

// All in one launch: the small gradients' loads fill the time in which the matrix
// instructions' blocks finish.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_gradients(Acts s, int m0, int Bn)
{
    __shared__ __attribute__((aligned(16))) float lds[2 * 40 * 64];
    const int m = m0 + blockIdx.y;
    const int block = blockIdx.x;
    if (block < IN_BLOCKS) input_gradient(s, m, block, Bn, lds);
    else if (block < IN_BLOCKS + DW_BLOCKS) weight_gradient(s, m, block - IN_BLOCKS, Bn);
    else bias_gradient(s, m, block - IN_BLOCKS - DW_BLOCKS, Bn, lds);
}

// Dense gradient of parameter p from the partial sums, each in order.
__device__ inline float gradient_of(const Acts &s, int m, int p, int nhead)
{
    float g = 0.0f;
    if (p >= HWT_SURR_W2 && p < HWT_SURR_B4 && !(p >= HWT_SURR_B2 && p < HWT_SURR_W3) &&
        !(p >= HWT_SURR_B3 && p < HWT_SURR_W4)) {
        const int l = p < HWT_SURR_B2 ? 2 : (p < HWT_SURR_B3 ? 3 : 4);
        const float *src = s.gw + ((size_t)m * 3 + (l - 2)) * DW_SPLIT * LAYER_W + (p - woff(l));
#pragma unroll
        for (int q = 0; q < DW_SPLIT; ++q) g += src[(size_t)q * LAYER_W];
        return g;
    }
    if (p < HWT_SURR_W5) {
        static_assert(HWT_SURR_W1 == 0 && HWT_SURR_B1 == HID * NIN && HWT_SURR_W2 == HWT_SURR_B1 + HID, "W1, b1 first");
        const int b = p < HWT_SURR_W2 ? p : p < HWT_SURR_W3 ? p - HWT_SURR_B2 + HWT_SURR_W2
                      : p < HWT_SURR_W4 ? p - HWT_SURR_B3 + HWT_SURR_W2 + HID : p - HWT_SURR_B4 + HWT_SURR_W2 + 2 * HID;
        const float *src = s.gs + (size_t)m * SMALL_PARTS * SMALL_N + b;
        return ((src[0] + src[SMALL_N]) + src[2 * SMALL_N]) + src[3 * SMALL_N];
    }
    // w5 and b5: a chain of adds over the tiles, its loads 32 at a time (one at a time
    // they were 100 us of a step)
    const float *src = s.hp + (size_t)m * (s.B / HEAD_ROWS) * (HID + 1) + (p - HWT_SURR_W5);
    constexpr int AHEAD = 32;
    for (int q = 0; q < nhead; q += AHEAD) {
        float v[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) v[k] = src[(size_t)min(q + k, nhead - 1) * (HID + 1)];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (q + k < nhead) g += v[k];
    }
    return g;
}

// Adam on parameter p of the FP32 masters; refreshes the BF16 copies (and
// transposes) of the 256x256 layers.
struct AdamArgs {
    float *m1, *m2;
    float lr, beta1, beta2, eps;
    float c1, c2;  // 1/(1-beta1^t), 1/(1-beta2^t)
};
__device__ inline void adam_step(const Net &net, const AdamArgs &a, int m, int p, float g)
{
    const size_t i = (size_t)m * PSTRIDE + p;
    const float mm = a.beta1 * a.m1[i] + (1.0f - a.beta1) * g;
    const float vv = a.beta2 * a.m2[i] + (1.0f - a.beta2) * g * g;
    a.m1[i] = mm;
    a.m2[i] = vv;
    const float w = net.P[i] - a.lr * (mm * a.c1) / (sqrtf(vv * a.c2) + a.eps);
    net.P[i] = w;
    int l = 0;
    if (p >= HWT_SURR_W2 && p < HWT_SURR_B2) l = 2;
    else if (p >= HWT_SURR_W3 && p < HWT_SURR_B3) l = 3;
    else if (p >= HWT_SURR_W4 && p < HWT_SURR_B4) l = 4;
    if (l) {
        const int idx = p - woff(l), nn = idx / HID, kk = idx % HID;
        const size_t base = ((size_t)m * 3 + (l - 2)) * LAYER_W;
        const uint16_t h = to_bf16(w);
        net.Wb[base + weight_at(nn, kk)] = h;
        net.WbT[base + weight_at(kk, nn)] = h;
    }
}

constexpr int PAR_BLOCKS = (NPAR + 255) / 256;
// The gradient of one evaluation, for callers who ask for it.
__global__ void k_grad_reduce(Acts s, int m0, int nhead)
{
    const int m = m0 + blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NPAR) s.g[(size_t)m * PSTRIDE + p] = gradient_of(s, m, p, nhead);
}

// Adam on a given gradient.
__global__ void k_adam(Net net, AdamArgs a, const float *__restrict__ grad)
{
    const int m = blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NPAR) adam_step(net, a, m, p, grad[(size_t)m * PSTRIDE + p]);
}

// A training step's: the gradient goes from its partial sums straight into Adam (17 us
// for four members; 116 us as two kernels, the head's chains one load at a time).  The
// head's chains are the longest, so their blocks start first.
__global__ __launch_bounds__(256) void k_update(Net net, AdamArgs a, Acts s, int nhead)
{
    const int m = blockIdx.y;
    const int p = (PAR_BLOCKS - 1 - blockIdx.x) * 256 + threadIdx.x;
    if (p < NPAR) adam_step(net, a, m, p, gradient_of(s, m, p, nhead));
}

// BF16 copies from the masters (after initialisation or a load).
__global__ void k_refresh_bf16(Net net, int members)
{
    const int m = blockIdx.y;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= members || idx >= 3 * LAYER_W) return;
    const int l = 2 + idx / LAYER_W, e = idx % LAYER_W, nn = e / HID, kk = e % HID;
    const uint16_t h = to_bf16(net.P[(size_t)m * PSTRIDE + woff(l) + e]);
    const size_t base = ((size_t)m * 3 + (l - 2)) * LAYER_W;
    net.Wb[base + weight_at(nn, kk)] = h;
    net.WbT[base + weight_at(kk, nn)] = h;
}

// --------------------------------------------------------------- inference
// One workgroup (4 waves) prices INF_ROWS = 128 options with every member.
// LDS holds the inputs and the BF16 activation tile act[row][neuron].  The
// hidden layers run as D = W A^T on the matrix cores: the weights are the
// A operand (loaded from L2, K-contiguous rows of W), the activations the B
// operand (LDS rows), so D[neuron][row] lands with four consecutive neurons
// of one row in each lane's accumulator quad and the epilogue writes them as
// one 8-byte store.  Wave w owns neurons [64w, 64w + 64) for all 128 rows,
// so each weight is read once per tile; a layer reads the whole tile, a
// barrier, then the epilogue overwrites it in place.  Layer 1 runs the same
// way on the FP32 matrix instructions (K = 8 in four 32x32x2 steps); every
// accumulator starts at its bias.  The output layer reduces per row across
// lanes and waves in a fixed order.  The yield curve is staged in LDS for the
// inputs.
// Bound by issue: 5.5 vector instructions a SiLU, two of them transcendental, keep
// the vector unit busy for 60% of the time and the matrix unit is for 47%, and the two
// hardly overlap.  (Neither wave priorities nor two tiles in one workgroup, one a step
// behind the other, changed that: 991 and 1075 us.)
constexpr int INF_YMAX = 256;  // keeps two 128-row tiles per CU in LDS

struct InferArgs {
    SOpts o;
    SYield y;
    Net net;
    int members;
    float threshold;
    double *out;       // prices (accepted options) or null
    double *mean;      // ensemble-mean price (predict) or null
    double *spread;    // member spread (predict) or null
    int8_t *in_box;    // (predict) or null
    int32_t *fb_idx;   // fallback list or null
    int32_t *fb_count; // [0] total, [1] out of box
    const int32_t *rows;      // option of each row (null: row i is option i)
    const int32_t *row_count; // number of listed rows (with `rows`)
};

// Accumulators of a wave's 2 x 4 blocks D[neuron][row] seeded with the
// layer's bias: lane l's value v belongs to neuron 32 mb + 8 (v/4) + 4 (l/32)
// + v%4 of the wave's 64, whatever the row block.
__device__ inline void bias_init(f32x16 (&acc)[2][4], const float *bias, int n0, int lane)
{
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
        f32x16 b;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 bv = *reinterpret_cast<const float4 *>(bias + n0 + 32 * mb + 8 * q + 4 * (lane >> 5));
            b[4 * q] = bv.x;
            b[4 * q + 1] = bv.y;
            b[4 * q + 2] = bv.z;
            b[4 * q + 3] = bv.w;
        }
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = b;
    }
}

// SiLU of the pre-activations, rounded to BF16, into the activation tile:
// the lane's four consecutive neurons of one row as one 8-byte store.
__device__ inline void silu_to_act(const f32x16 (&acc)[2][4], uint16_t *act, int n0, int lane)
{
    const int mrow = lane & 31;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = n0 + 32 * mb + 8 * q + 4 * (lane >> 5);
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                const f32x16 &a = acc[mb][nb];
                const uint2 pk = make_uint2(pack_bf16x2(silu(a[4 * q]), silu(a[4 * q + 1])),
                                            pack_bf16x2(silu(a[4 * q + 2]), silu(a[4 * q + 3])));
                *reinterpret_cast<uint2 *>(act + (32 * nb + mrow) * ACT_LD + col) = pk;
            }
        }
}

// A wave's weights of one layer (two blocks of 32 neurons), INF_AHEAD of the 16
// k-steps in flight, the first of the next layer during a layer's epilogue (475,000
// rows: 1085 us without, 987; 3 or 4 steps ahead spill, 1000 and 1028).
constexpr int INF_AHEAD = 2;
struct InferWeights {
    bf16x8 w[INF_AHEAD][2];
    const uint16_t *p;
    __device__ void start(const uint16_t *W, int n0, int lane)
    {
        p = W + ((size_t)(n0 >> 5) * (HID / 16) * 64 + lane) * 8;
#pragma unroll
        for (int k = 0; k < INF_AHEAD; ++k) load(k);
    }
    __device__ void load(int k)
    {
        w[k % INF_AHEAD][0] = load_frag(p + k * 64 * 8);
        w[k % INF_AHEAD][1] = load_frag(p + (HID / 16 + k) * 64 * 8);
    }
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_infer(InferArgs g)
{
    static_assert(INF_ROWS == 128, "the layer-1 and head mappings assume 128 rows per tile");
    __shared__ __attribute__((aligned(16))) uint16_t act[INF_ROWS * ACT_LD];
    __shared__ float xs[INF_ROWS * NIN];
    __shared__ double bases[INF_ROWS];
    __shared__ float hp[4 * INF_ROWS];
    __shared__ float ysum[INF_ROWS], ymin[INF_ROWS], ymax[INF_ROWS];
    __shared__ int32_t okf[INF_ROWS];
    __shared__ int32_t fb_local[INF_ROWS];
    __shared__ int32_t fb_n, fb_out, fb_base;
    // the curve, while the inputs are made; then each member's b2..b4 and w5
    __shared__ __attribute__((aligned(16))) char front[4 * HID * 4];
    static_assert(INF_YMAX * 12 <= (int)sizeof(front), "the curve fits");
    double *yr = reinterpret_cast<double *>(front);
    int32_t *yd = reinterpret_cast<int32_t *>(front + INF_YMAX * 8);
    float *vec = reinterpret_cast<float *>(front);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int r0 = blockIdx.x * INF_ROWS;
    const int nrows = g.rows ? *g.row_count : g.o.n;
    if (r0 >= nrows) return;  // the whole tile is past the listed rows

    // curves that fit are read from LDS, by binary search when their days
    // never decrease; both lookups give the reference's value
    const bool staged = g.y.n <= INF_YMAX;
    int unsorted = 0;
    if (staged) {
        for (int k = t; k < g.y.n; k += 256) {
            yr[k] = g.y.rate[k];
            yd[k] = g.y.day[k];
            if (k + 1 < g.y.n && g.y.day[k] > g.y.day[k + 1]) unsorted = 1;
        }
    }
    // unconditional barrier: it also orders the LDS writes below after every
    // thread's curve staging, whatever the curve's length
    const int any_unsorted = __syncthreads_or(unsorted);
    const bool sorted = staged && !any_unsorted;
    if (t < INF_ROWS) {
        const int i = r0 + t < nrows ? (g.rows ? g.rows[r0 + t] : r0 + t) : -1;
        float x[NIN] = {};
        double base = 0.0;
        const bool ok = i >= 0 && surr_inputs(g.o, i, x, base, [&](double tt, int tu) {
            return sorted ? yield_at_sorted(tt, tu, yr, yd, g.y.n) : yield_at(tt, tu, g.y.rate, g.y.day, g.y.n);
        });
#pragma unroll
        for (int k = 0; k < NIN; ++k) xs[t * NIN + k] = x[k];
        bases[t] = base;
        okf[t] = ok;
        ysum[t] = 0.0f;
        ymin[t] = INFINITY;
        ymax[t] = -INFINITY;
    }
    if (t == 0) fb_n = fb_out = 0;
    __syncthreads();

    const int mrow = lane & 31, khalf = 8 * (lane >> 5);
    const int n0 = wave * 64;  // this wave's output neurons in the hidden layers
    InferWeights w;
    w.start(g.net.Wb, n0, lane);
    for (int m = 0; m < g.members; ++m) {
        const float *P = g.net.P + (size_t)m * PSTRIDE;
        // the member's vectors into LDS, requested beside layer 1's (each layer
        // fetching its own from L2 waited for it)
        float own[4];
#pragma unroll
        for (int l = 2; l <= 4; ++l) own[l - 2] = P[boff(l) + t];
        own[3] = P[HWT_SURR_W5 + t];
        // layer 1 (FP32 MFMA 32x32x2, K = 8 in four steps): D[neuron][row] =
        // b1 + W1 x^T, with the lane's A value W1[n][k] and B value x[row][k]
        {
            f32x16 acc[2][4];
            bias_init(acc, P + HWT_SURR_B1, n0, lane);
#pragma unroll
            for (int k = 0; k < NIN; k += 2) {
                const int kk = k + (lane >> 5);
                const float a0 = P[HWT_SURR_W1 + (n0 + mrow) * NIN + kk];
                const float a1 = P[HWT_SURR_W1 + (n0 + 32 + mrow) * NIN + kk];
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    const float bx = xs[(32 * nb + mrow) * NIN + kk];
                    acc[0][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, bx, acc[0][nb], 0, 0, 0);
                    acc[1][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, bx, acc[1][nb], 0, 0, 0);
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) vec[k * HID + t] = own[k];
            silu_to_act(acc, act, n0, lane);
        }
        __syncthreads();
        for (int l = 2; l <= 4; ++l) {
            const uint16_t *ab = act + mrow * ACT_LD + khalf;
            f32x16 acc[2][4];
            bias_init(acc, vec + (l - 2) * HID, n0, lane);
#pragma unroll
            for (int k = 0; k < HID / 16; ++k) {
                const bf16x8 a0 = w.w[k % INF_AHEAD][0], a1 = w.w[k % INF_AHEAD][1];
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    const bf16x8 b = load_frag(ab + nb * 32 * ACT_LD + 16 * k);
                    acc[0][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b, acc[0][nb], 0, 0, 0);
                    acc[1][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b, acc[1][nb], 0, 0, 0);
                }
                if (k + INF_AHEAD < HID / 16) w.load(k + INF_AHEAD);
                __builtin_amdgcn_sched_barrier(0);  // reads no further ahead: registers are full
            }
            // the next layer's first weights, during this one's epilogue (the last
            // member's last: its own again)
            w.start(g.net.Wb + ((size_t)min(l < 4 ? m : m + 1, g.members - 1) * 3 + (l < 4 ? l - 1 : 0)) * LAYER_W, n0, lane);
            __syncthreads();  // every wave has read this layer's input tile
            if (l < 4) {
                silu_to_act(acc, act, n0, lane);
                __syncthreads();
            } else {
                // output layer in FP32 from the accumulators: per row, the
                // lane's 32 neurons, then the lane pair holding the same row,
                // then the four waves
                float p[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int col = n0 + 32 * mb + 8 * q + 4 * (lane >> 5);
                        const float4 w5 = *reinterpret_cast<const float4 *>(vec + 3 * HID + col);
#pragma unroll
                        for (int nb = 0; nb < 4; ++nb) {
                            const f32x16 &a = acc[mb][nb];
                            p[nb] = fmaf(w5.x, silu(a[4 * q]), p[nb]);
                            p[nb] = fmaf(w5.y, silu(a[4 * q + 1]), p[nb]);
                            p[nb] = fmaf(w5.z, silu(a[4 * q + 2]), p[nb]);
                            p[nb] = fmaf(w5.w, silu(a[4 * q + 3]), p[nb]);
                        }
                    }
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    const float v = p[nb] + __shfl_xor(p[nb], 32, 64);
                    if (lane < 32) hp[wave * INF_ROWS + 32 * nb + lane] = v;
                }
                __syncthreads();
                if (t < INF_ROWS) {
                    const float yv = ((hp[t] + hp[INF_ROWS + t]) + (hp[2 * INF_ROWS + t] + hp[3 * INF_ROWS + t])) +
                                     P[HWT_SURR_B5];
                    ysum[t] += yv;
                    ymin[t] = fminf(ymin[t], yv);
                    ymax[t] = fmaxf(ymax[t], yv);
                }
            }
        }
    }
    if (t < INF_ROWS) {
        const int i = r0 + t < nrows ? (g.rows ? g.rows[r0 + t] : r0 + t) : -1;
        if (i >= 0) {
            const double mean = bases[t] + RES * (double)(ysum[t] / (float)g.members);
            const double spread = RES * (double)(ymax[t] - ymin[t]);
            const bool ok = okf[t] != 0;
            if (g.mean) g.mean[i] = ok ? mean : NAN;
            if (g.spread) g.spread[i] = ok ? spread : NAN;
            if (g.in_box) g.in_box[i] = (int8_t)ok;
            // a non-finite member output makes the mean non-finite while
            // fminf/fmaxf would drop it from the spread: never accepted
            const bool accept = ok && isfinite(mean) && spread <= (double)g.threshold;
            if (g.out && accept) g.out[i] = mean;
            if (g.fb_idx && !accept) {
                fb_local[atomicAdd(&fb_n, 1)] = i;
                if (!ok) atomicAdd(&fb_out, 1);
            }
        }
    }
    if (g.fb_idx) {
        __syncthreads();
        if (t == 0 && fb_n > 0) {
            fb_base = atomicAdd(&g.fb_count[0], fb_n);
            atomicAdd(&g.fb_count[1], fb_out);
        }
        __syncthreads();
        if (t < fb_n) g.fb_idx[fb_base + t] = fb_local[t];
    }
}

// Splits a batch before inference: options outside the training box go to
// the fallback list (fb_idx, fb_count[0] and [1]), the others to the row list
// of the inference kernel (rows, row_count).  A block takes BOX_CHUNK options
// and stages both lists in LDS, so the global counters see one atomic per
// list per block (same-address atomics serialise in L2: one per 256 options
// cost more than the whole test).  Order inside the lists is arbitrary.
// A wave takes its places in a staged list with one LDS atomic: 4,096 a block on two
// addresses took most of its time (500,000 options: 27 us with 256 threads, now 13.5;
// chunks of 2,048 15 us, of 1,024 25: the lists' heads).
constexpr int BOX_CHUNK = 4096, BOX_THREADS = 1024;

__global__ __launch_bounds__(BOX_THREADS) void k_box(SOpts o, int32_t *__restrict__ fb_idx, int32_t *__restrict__ fb_count,
                                             int32_t *__restrict__ rows, int32_t *__restrict__ row_count)
{
    __shared__ int32_t nin, nout, bin, bout;
    __shared__ int32_t lin[BOX_CHUNK], lout[BOX_CHUNK];
    const int t = threadIdx.x, i0 = blockIdx.x * BOX_CHUNK;
    if (t == 0) nin = nout = 0;
    __syncthreads();
    const int lane = t & 63;
    const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
    for (int k = 0; k < BOX_CHUNK / BOX_THREADS; ++k) {
        // the parameter test alone; a listed option that still fails the tree
        // test is sent to the fallback list by the inference kernel
        const int i = i0 + t + BOX_THREADS * k;
        const bool in = i < o.n && surr_param_box(o, i), off = i < o.n && !in;
        const unsigned long long mi = __ballot(in), mo = __ballot(off);
        int pi = 0, po = 0;
        if (lane == 0) {
            if (mi) pi = atomicAdd(&nin, (int)__popcll(mi));
            if (mo) po = atomicAdd(&nout, (int)__popcll(mo));
        }
        pi = __builtin_amdgcn_readfirstlane(pi);
        po = __builtin_amdgcn_readfirstlane(po);
        if (in) lin[pi + __popcll(mi & below)] = i;
        if (off) lout[po + __popcll(mo & below)] = i;
    }
    __syncthreads();
    if (t == 0) {
        bin = nin ? atomicAdd(row_count, nin) : 0;
        bout = nout ? atomicAdd(&fb_count[0], nout) : 0;
        if (nout) atomicAdd(&fb_count[1], nout);
    }
    __syncthreads();
    for (int k = t; k < nin; k += BOX_THREADS) rows[bin + k] = lin[k];
    for (int k = t; k < nout; k += BOX_THREADS) fb_idx[bout + k] = lout[k];
}

// The start of a pass: its counters to zero and the device's constant-rate wall clock
// into stamp 0.  Stamps mark a pass's parts, which events cannot give inside a graph:
// 1 as the gather starts, 2 as the last of the scatter's blocks ends (kernels of their
// own took 4 us each).
__global__ void k_begin_pass(int32_t *count, uint64_t *stamps)
{
    if (threadIdx.x < 8) count[threadIdx.x] = 0;
    if (threadIdx.x == 0) stamps[0] = stamps[1] = stamps[2] = __builtin_amdgcn_s_memrealtime();
}

// Fallback list -> compact option arrays, and prices back to input order.
struct Compact {
    double *strike, *maturity, *length, *a, *sigma;
    uint16_t *tu, *steps;
    int8_t *type;
};

__global__ void k_fb_gather(SOpts o, const int32_t *__restrict__ idx, const int32_t *__restrict__ count, Compact c,
                            uint64_t *__restrict__ stamps)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j == 0) stamps[1] = __builtin_amdgcn_s_memrealtime();
    if (j >= count[0]) return;
    const int i = idx[j];
    c.strike[j] = o.strike[i];
    c.maturity[j] = o.maturity[i];
    c.length[j] = o.length[i];
    c.a[j] = o.a[i];
    c.sigma[j] = o.sigma[i];
    c.tu[j] = o.tu[i];
    c.steps[j] = o.steps[i];
    c.type[j] = o.type[i];
}

__global__ void k_fb_scatter(const int32_t *__restrict__ idx, const int32_t *__restrict__ count,
                             const double *__restrict__ tmp, double *__restrict__ out, uint64_t *__restrict__ stamps)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x, n = count[0];
    if (j < n) out[idx[j]] = tmp[j];
    if (threadIdx.x == 0 && (j < n || j == 0))
        atomicMax(reinterpret_cast<unsigned long long *>(stamps + 2), (unsigned long long)__builtin_amdgcn_s_memrealtime());
}

__global__ void k_zero_i32(int32_t *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_zero_f64(double *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

int fail(int code, const std::string &msg) { return hwt_internal_fail(code, msg.c_str()); }

#define SURR_HIP(call)                                                                         \
    do {                                                                                       \
        hipError_t err_ = (call);                                                              \
        if (err_ != hipSuccess)                                                                \
            return fail(HWT_EHIP, std::string(#call) + ": " + hipGetErrorString(err_));        \
    } while (0)

bool valid_opts(const hwt_options_f64 *o)
{
    return o && o->n >= 0 &&
           (o->n == 0 || (o->strike && o->maturity && o->length && o->term_unit && o->term_steps && o->a &&
                          o->sigma && o->type));
}
bool valid_yield(const hwt_yield_f64 *y) { return y && y->n > 0 && y->rate && y->day; }

} // namespace

struct hwt_surrogate {
    int device = 0;
    hipStream_t stream = nullptr;
    hwt_surr_config cfg{};
    int members = 4, B = 8192;
    int32_t train_cap = 0, infer_cap = 0, ycap = 0;
    int32_t ntrain = 0;
    int64_t step = 0;
    int epochs_done = 0;
    std::mt19937_64 rng;
    // device
    void *mem = nullptr;
    size_t bytes = 0;
    Net net{};
    Acts acts{};
    float *m1 = nullptr, *m2 = nullptr;
    float *X = nullptr, *target = nullptr;
    int32_t *perm = nullptr;  // [members][train_cap]
    int32_t *rows = nullptr;  // test hook rows [B]
    int32_t *bad = nullptr;
    int32_t *fb_idx = nullptr;   // fallback list: out-of-box options, then uncertain in-box ones
    int32_t *inf_rows = nullptr; // in-box options, the rows of the inference kernel
    int32_t *fb_count = nullptr; // [0] fallback total, [1] of which out of box, [4] inference rows;
                                 // [8..13] three u64 wall-clock stamps of a pricing pass
    double *fb_tmp = nullptr;
    Compact comp{};
    int32_t *h_count = nullptr;  // pinned copy of fb_count [16]
    int wall_khz = 100000;       // rate of the device's constant wall clock
    double *h_loss = nullptr;    // pinned [members]
    hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr;
    // the pricing pass captured as one graph, and the arguments it was
    // captured with
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    struct PassKey {
        hwt_options_f64 o;
        hwt_yield_f64 y;
        double *out;
        const hwt_plan *tree;
        uint64_t tree_serial;
        float threshold;
        int32_t members;
    } key{};
};

namespace {

// Forward + backward of members [m0, m0+mc) on the gathered rows; leaves the
// gradient's partial sums in acts.
int forward_backward(hwt_surrogate *s, int m0, int mc, int Bn)
{
    k_train_tile<<<dim3(Bn / TILE_ROWS, mc), 512, 0, s->stream>>>(s->net, s->acts, m0, Bn);
    k_gradients<<<dim3(IN_BLOCKS + DW_BLOCKS + BIAS_BLOCKS, mc), 256, 0, s->stream>>>(s->acts, m0, Bn);
    SURR_HIP(hipGetLastError());
    return HWT_OK;
}

float lr_at(const hwt_surrogate *s, int64_t step, int64_t total)
{
    const hwt_surr_config &c = s->cfg;
    const double warm = std::max<double>(1.0, c.warmup_frac * (double)total);
    if (step < warm) return (float)(c.lr_max * (step + 1) / warm);
    const double f = std::min(1.0, (step - warm) / std::max(1.0, (double)total - warm));
    return (float)(c.lr_min + 0.5 * (c.lr_max - c.lr_min) * (1.0 + std::cos(M_PI * f)));
}

// Adam on the gradient in acts.g, or on the partial sums a step over nhead head
// blocks has left in acts.
int adam_launch(hwt_surrogate *s, float lr, int nhead)
{
    const hwt_surr_config &c = s->cfg;
    const double t = (double)(s->step + 1);
    const AdamArgs a{s->m1, s->m2, lr, c.beta1, c.beta2, c.eps,
                     (float)(1.0 / (1.0 - std::pow((double)c.beta1, t))),
                     (float)(1.0 / (1.0 - std::pow((double)c.beta2, t)))};
    const dim3 grid(PAR_BLOCKS, s->members);
    if (nhead) k_update<<<grid, 256, 0, s->stream>>>(s->net, a, s->acts, nhead);
    else k_adam<<<grid, 256, 0, s->stream>>>(s->net, a, s->acts.g);
    SURR_HIP(hipGetLastError());
    ++s->step;
    return HWT_OK;
}

void init_params(hwt_surrogate *s, std::vector<float> &P)
{
    // PyTorch-style uniform init: U(-1/sqrt(fan_in), 1/sqrt(fan_in)) for weights and biases
    P.assign((size_t)s->members * PSTRIDE, 0.0f);
    for (int m = 0; m < s->members; ++m) {
        std::mt19937_64 g(s->cfg.seed * 1000003ull + 7919ull * (uint64_t)m + 1ull);
        auto fill = [&](int off, int count, int fan_in) {
            std::uniform_real_distribution<float> U(-1.0f / std::sqrt((float)fan_in), 1.0f / std::sqrt((float)fan_in));
            for (int i = 0; i < count; ++i) P[(size_t)m * PSTRIDE + off + i] = U(g);
        };
        fill(HWT_SURR_W1, HID * NIN, NIN);
        fill(HWT_SURR_B1, HID, NIN);
        for (int l = 2; l <= 4; ++l) {
            fill(woff(l), LAYER_W, HID);
            fill(boff(l), HID, HID);
        }
        fill(HWT_SURR_W5, HID, HID);
        fill(HWT_SURR_B5, 1, HID);
    }
}

struct DeviceGuardS {
    int prev = -1;
    explicit DeviceGuardS(int dev)
    {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        if (prev != dev) (void)hipSetDevice(dev);
    }
    ~DeviceGuardS()
    {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

} // namespace

extern "C" {

void hwt_surr_config_init(hwt_surr_config *c)
{
    if (!c) return;
    std::memset(c, 0, sizeof(*c));
    c->members = 4;
    c->batch = 8192;
    c->lr_max = 2e-3f;
    c->lr_min = 2e-5f;
    c->warmup_frac = 0.02f;
    c->beta1 = 0.9f;
    c->beta2 = 0.999f;
    c->eps = 1e-8f;
    c->spread_threshold = 1e-3f;
    c->seed = 1;
}

void hwt_surr_destroy(hwt_surrogate *s)
{
    if (!s) return;
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    if (s->mem) (void)hipFree(s->mem);
    if (s->h_count) (void)hipHostFree(s->h_count);
    if (s->h_loss) (void)hipHostFree(s->h_loss);
    for (hipEvent_t e : {s->e0, s->e1, s->e2})
        if (e) (void)hipEventDestroy(e);
    if (s->exec) (void)hipGraphExecDestroy(s->exec);
    if (s->graph) (void)hipGraphDestroy(s->graph);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
}

int hwt_surr_create(hwt_surrogate **out, int32_t train_capacity, int32_t infer_capacity, int32_t yield_capacity,
                    const hwt_surr_config *cfg)
{
    if (!out || train_capacity < 0 || infer_capacity < 0 || yield_capacity < 1)
        return fail(HWT_EINVAL, "hwt_surr_create: bad arguments");
    *out = nullptr;
    hwt_surrogate *s = new (std::nothrow) hwt_surrogate();
    if (!s) return fail(HWT_ENOMEM, "hwt_surr_create: host allocation");
    if (cfg) s->cfg = *cfg;
    else hwt_surr_config_init(&s->cfg);
    const hwt_surr_config &c = s->cfg;
    if (c.members < 1 || c.members > HWT_SURR_MAX_MEMBERS || c.batch < BATCH_STEP || c.batch % BATCH_STEP != 0 ||
        c.batch > (1 << 20) || !(c.lr_max > 0.0f) || !(c.beta1 >= 0.0f && c.beta1 < 1.0f) ||
        !(c.beta2 >= 0.0f && c.beta2 < 1.0f) || !(c.eps > 0.0f) || !(c.spread_threshold >= 0.0f)) {
        delete s;
        return fail(HWT_EINVAL, "hwt_surr_create: bad configuration");
    }
    s->members = c.members;
    s->B = c.batch;
    s->train_cap = train_capacity;
    s->infer_cap = infer_capacity;
    s->ycap = yield_capacity;
    s->rng.seed(c.seed * 2654435761ull + 12345ull);
    auto bail = [&](int code, const std::string &msg) {
        hwt_surr_destroy(s);
        return fail(code, msg);
    };
    if (hipGetDevice(&s->device) != hipSuccess) return bail(HWT_EHIP, "hipGetDevice failed");
    if (hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(HWT_EHIP, "hipStreamCreate failed");
    for (hipEvent_t *e : {&s->e0, &s->e1, &s->e2})
        if (hipEventCreate(e) != hipSuccess) return bail(HWT_EHIP, "hipEventCreate failed");
    {
        int khz = 0;
        if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, s->device) == hipSuccess && khz > 0)
            s->wall_khz = khz;
        (void)hipGetLastError();
    }
    const size_t M = s->members, B = s->B, T = std::max(train_capacity, 1), I = std::max(infer_capacity, 1);
    size_t off = 0;
    auto carve = [&](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~(size_t)255;
        return at;
    };
    const size_t oP = carve(M * PSTRIDE * 4), oWb = carve(M * 3 * LAYER_W * 2), oWbT = carve(M * 3 * LAYER_W * 2);
    const size_t om1 = carve(M * PSTRIDE * 4), om2 = carve(M * PSTRIDE * 4);
    const size_t oxb = carve(M * B * NIN * 4), otb = carve(M * B * 4);
    const size_t oaT = carve(M * 3 * B * HID * 2), odzT = carve(M * 3 * B * HID * 2), odz1 = carve(M * HID * B * 4);
    const size_t oy = carve(M * B * 4), ogw = carve(M * 3 * DW_SPLIT * LAYER_W * 4), ogs = carve(M * SMALL_PARTS * SMALL_N * 4);
    const size_t ohp = carve(M * (B / HEAD_ROWS) * (HID + 1) * 4), oloss = carve(M * 8), og = carve(M * PSTRIDE * 4);
    const size_t oX = carve(T * NIN * 4), otg = carve(T * 4), operm = carve(M * T * 4), orows = carve(B * 4);
    const size_t obad = carve(4), ofbi = carve(I * 4), ofbc = carve(16 * 4), ofbt = carve(I * 8);
    const size_t oinr = carve(I * 4);
    const size_t ocs = carve(I * 8), ocm = carve(I * 8), ocl = carve(I * 8), oca = carve(I * 8), ocg = carve(I * 8);
    const size_t ocu = carve(I * 2), ocst = carve(I * 2), octy = carve(I);
    s->bytes = off;
    hipError_t em = hipMalloc(&s->mem, s->bytes);
    if (em != hipSuccess) {  // again, with the idle one-shot workspaces given back
        (void)hipGetLastError();
        hwt_trim();
        em = hipMalloc(&s->mem, s->bytes);
    }
    if (em != hipSuccess) return bail(HWT_ENOMEM, "hipMalloc surrogate workspace failed");
    char *b = (char *)s->mem;
    s->net.P = (float *)(b + oP);
    s->net.Wb = (uint16_t *)(b + oWb);
    s->net.WbT = (uint16_t *)(b + oWbT);
    s->m1 = (float *)(b + om1);
    s->m2 = (float *)(b + om2);
    Acts &a = s->acts;
    a.B = (int)B;
    a.xb = (float *)(b + oxb);
    a.tb = (float *)(b + otb);
    a.aT = (uint16_t *)(b + oaT);
    a.dzT = (uint16_t *)(b + odzT);
    a.dz1 = (float *)(b + odz1);
    a.y = (float *)(b + oy);
    a.gw = (float *)(b + ogw);
    a.gs = (float *)(b + ogs);
    a.hp = (float *)(b + ohp);
    a.loss = (double *)(b + oloss);
    a.g = (float *)(b + og);
    s->X = (float *)(b + oX);
    s->target = (float *)(b + otg);
    s->perm = (int32_t *)(b + operm);
    s->rows = (int32_t *)(b + orows);
    s->bad = (int32_t *)(b + obad);
    s->fb_idx = (int32_t *)(b + ofbi);
    s->inf_rows = (int32_t *)(b + oinr);
    s->fb_count = (int32_t *)(b + ofbc);
    s->fb_tmp = (double *)(b + ofbt);
    s->comp = Compact{(double *)(b + ocs), (double *)(b + ocm), (double *)(b + ocl), (double *)(b + oca),
                      (double *)(b + ocg), (uint16_t *)(b + ocu), (uint16_t *)(b + ocst), (int8_t *)(b + octy)};
    if (hipHostMalloc((void **)&s->h_count, 16 * sizeof(int32_t), 0) != hipSuccess ||
        hipHostMalloc((void **)&s->h_loss, M * sizeof(double), 0) != hipSuccess)
        return bail(HWT_ENOMEM, "hipHostMalloc failed");
    // zero everything once (gradient partials of unused rows stay defined)
    if (hipMemsetAsync(s->mem, 0, s->bytes, s->stream) != hipSuccess) return bail(HWT_EHIP, "hipMemsetAsync failed");
    std::vector<float> P;
    init_params(s, P);
    if (hipMemcpyAsync(s->net.P, P.data(), P.size() * 4, hipMemcpyHostToDevice, s->stream) != hipSuccess)
        return bail(HWT_EHIP, "hipMemcpy parameters failed");
    k_refresh_bf16<<<dim3((3 * LAYER_W + 255) / 256, s->members), 256, 0, s->stream>>>(s->net, s->members);
    if (hipStreamSynchronize(s->stream) != hipSuccess) return bail(HWT_EHIP, "initialisation failed");
    *out = s;
    return HWT_OK;
}

int hwt_surr_set_training_data(hwt_surrogate *s, const hwt_options_f64 *o, const hwt_yield_f64 *y, const double *prices)
{
    if (!s || !valid_opts(o) || !valid_yield(y) || (o->n > 0 && !prices))
        return fail(HWT_EINVAL, "hwt_surr_set_training_data: null or negative-size argument");
    if (o->n > s->train_cap) return fail(HWT_ENOMEM, "hwt_surr_set_training_data: more samples than the capacity");
    if (o->n < s->B) return fail(HWT_EINVAL, "hwt_surr_set_training_data: fewer samples than one batch");
    DeviceGuardS dg(s->device);
    k_zero_i32<<<1, 32, 0, s->stream>>>(s->bad, 1);
    k_train_inputs<<<(o->n + 255) / 256, 256, 0, s->stream>>>(sopts(*o), SYield{y->n, y->rate, y->day}, prices, s->X,
                                                              s->target, s->bad);
    SURR_HIP(hipMemcpyAsync(s->h_count, s->bad, 4, hipMemcpyDeviceToHost, s->stream));
    SURR_HIP(hipStreamSynchronize(s->stream));
    if (s->h_count[0] > 0)
        return fail(HWT_EINVAL, std::to_string(s->h_count[0]) + " training sample(s) outside the training box");
    s->ntrain = o->n;
    return HWT_OK;
}

int hwt_surr_train(hwt_surrogate *s, int32_t epochs, int32_t total_epochs, hwt_surr_stats *stats)
{
    if (!s || epochs < 0 || total_epochs < s->epochs_done + epochs)
        return fail(HWT_EINVAL, "hwt_surr_train: bad arguments");
    if (s->ntrain < s->B) return fail(HWT_EINVAL, "hwt_surr_train: no training data");
    DeviceGuardS dg(s->device);
    const int spe = s->ntrain / s->B;  // steps per epoch (the remainder rotates through the shuffles)
    const int64_t total = (int64_t)total_epochs * spe;
    std::vector<int32_t> perm((size_t)s->members * s->ntrain);
    SURR_HIP(hipEventRecord(s->e0, s->stream));
    for (int ep = 0; ep < epochs; ++ep) {
        for (int m = 0; m < s->members; ++m) {
            int32_t *p = perm.data() + (size_t)m * s->ntrain;
            for (int i = 0; i < s->ntrain; ++i) p[i] = i;
            for (int i = s->ntrain - 1; i > 0; --i) {
                const int j = (int)(s->rng() % (uint64_t)(i + 1));
                std::swap(p[i], p[j]);
            }
        }
        SURR_HIP(hipStreamSynchronize(s->stream));  // the previous epoch's reads of perm are done
        SURR_HIP(hipMemcpyAsync(s->perm, perm.data(), perm.size() * 4, hipMemcpyHostToDevice, s->stream));
        k_zero_f64<<<1, 64, 0, s->stream>>>(s->acts.loss, s->members);
        for (int it = 0; it < spe; ++it) {
            k_gather<<<dim3(s->B / 256 + (s->B % 256 != 0), s->members), 256, 0, s->stream>>>(
                s->X, s->target, s->perm, s->ntrain, (int64_t)it * s->B, s->B, s->B, s->acts.xb, s->acts.tb, 0);
            const int rc = forward_backward(s, 0, s->members, s->B);
            if (rc) return rc;
            const int arc = adam_launch(s, lr_at(s, s->step, total), s->B / HEAD_ROWS);
            if (arc) return arc;
        }
        ++s->epochs_done;
    }
    SURR_HIP(hipEventRecord(s->e1, s->stream));
    SURR_HIP(hipMemcpyAsync(s->h_loss, s->acts.loss, s->members * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    SURR_HIP(hipStreamSynchronize(s->stream));
    if (stats) {
        std::memset(stats, 0, sizeof(*stats));
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, s->e0, s->e1) == hipSuccess) stats->ms = ms;
        double l = 0.0;
        for (int m = 0; m < s->members; ++m) l += s->h_loss[m];
        stats->loss = epochs > 0 ? l / ((double)s->members * spe * s->B) : 0.0;
        stats->steps = s->step;
    }
    return HWT_OK;
}

int hwt_surr_eval_rows(hwt_surrogate *s, int32_t member, const int32_t *host_rows, int32_t n, float *host_out,
                       float *host_loss, float *host_grad)
{
    if (!s || member < 0 || member >= s->members || !host_rows || n < BATCH_STEP || n % BATCH_STEP != 0 || n > s->B)
        return fail(HWT_EINVAL, "hwt_surr_eval_rows: bad arguments");
    for (int i = 0; i < n; ++i)
        if (host_rows[i] < 0 || host_rows[i] >= s->ntrain) return fail(HWT_EINVAL, "hwt_surr_eval_rows: row out of range");
    DeviceGuardS dg(s->device);
    // Rows go into the member's slot of the batch buffers; the kernels use the
    // batch pitch s->B and the actual row count n.
    SURR_HIP(hipMemcpyAsync(s->rows, host_rows, (size_t)n * 4, hipMemcpyHostToDevice, s->stream));
    k_gather<<<dim3((n + 255) / 256, 1), 256, 0, s->stream>>>(s->X, s->target, s->rows, 0, 0, n, s->B, s->acts.xb,
                                                              s->acts.tb, member);
    k_zero_f64<<<1, 64, 0, s->stream>>>(s->acts.loss, s->members);
    const int rc = forward_backward(s, member, 1, n);
    if (rc) return rc;
    if (host_grad) {
        k_grad_reduce<<<dim3(PAR_BLOCKS, 1), 256, 0, s->stream>>>(s->acts, member, n / HEAD_ROWS);
        SURR_HIP(hipGetLastError());
    }
    SURR_HIP(hipMemcpyAsync(s->h_loss, s->acts.loss, s->members * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    if (host_out)
        SURR_HIP(hipMemcpyAsync(host_out, s->acts.y + (size_t)member * s->B, (size_t)n * 4, hipMemcpyDeviceToHost,
                                s->stream));
    if (host_grad)
        SURR_HIP(hipMemcpyAsync(host_grad, s->acts.g + (size_t)member * PSTRIDE, (size_t)NPAR * 4,
                                hipMemcpyDeviceToHost, s->stream));
    SURR_HIP(hipStreamSynchronize(s->stream));
    if (host_loss) *host_loss = (float)(s->h_loss[member] / n);
    return HWT_OK;
}

int hwt_surr_get_inputs(hwt_surrogate *s, const int32_t *host_rows, int32_t n, float *host_x, float *host_target)
{
    if (!s || !host_rows || n < 0) return fail(HWT_EINVAL, "hwt_surr_get_inputs: bad arguments");
    DeviceGuardS dg(s->device);
    std::vector<float> X((size_t)s->ntrain * NIN), t(s->ntrain);
    SURR_HIP(hipMemcpy(X.data(), s->X, X.size() * 4, hipMemcpyDeviceToHost));
    SURR_HIP(hipMemcpy(t.data(), s->target, t.size() * 4, hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i) {
        const int r = host_rows[i];
        if (r < 0 || r >= s->ntrain) return fail(HWT_EINVAL, "hwt_surr_get_inputs: row out of range");
        if (host_x) std::memcpy(host_x + (size_t)i * NIN, X.data() + (size_t)r * NIN, NIN * 4);
        if (host_target) host_target[i] = t[r];
    }
    return HWT_OK;
}

int hwt_surr_adam_step(hwt_surrogate *s, const float *host_grad, float lr)
{
    if (!s || !host_grad || !(lr >= 0.0f)) return fail(HWT_EINVAL, "hwt_surr_adam_step: bad arguments");
    DeviceGuardS dg(s->device);
    for (int m = 0; m < s->members; ++m)
        SURR_HIP(hipMemcpyAsync(s->acts.g + (size_t)m * PSTRIDE, host_grad + (size_t)m * NPAR, (size_t)NPAR * 4,
                                hipMemcpyHostToDevice, s->stream));
    const int rc = adam_launch(s, lr, 0);
    if (rc) return rc;
    SURR_HIP(hipStreamSynchronize(s->stream));
    return HWT_OK;
}

int hwt_surr_get_params(hwt_surrogate *s, float *host)
{
    if (!s || !host) return fail(HWT_EINVAL, "hwt_surr_get_params: bad arguments");
    DeviceGuardS dg(s->device);
    SURR_HIP(hipStreamSynchronize(s->stream));
    for (int m = 0; m < s->members; ++m)
        SURR_HIP(hipMemcpy(host + (size_t)m * NPAR, s->net.P + (size_t)m * PSTRIDE, (size_t)NPAR * 4,
                           hipMemcpyDeviceToHost));
    return HWT_OK;
}

int hwt_surr_set_params(hwt_surrogate *s, const float *host)
{
    if (!s || !host) return fail(HWT_EINVAL, "hwt_surr_set_params: bad arguments");
    DeviceGuardS dg(s->device);
    SURR_HIP(hipStreamSynchronize(s->stream));
    for (int m = 0; m < s->members; ++m)
        SURR_HIP(hipMemcpy(s->net.P + (size_t)m * PSTRIDE, host + (size_t)m * NPAR, (size_t)NPAR * 4,
                           hipMemcpyHostToDevice));
    k_refresh_bf16<<<dim3((3 * LAYER_W + 255) / 256, s->members), 256, 0, s->stream>>>(s->net, s->members);
    SURR_HIP(hipGetLastError());
    SURR_HIP(hipStreamSynchronize(s->stream));
    return HWT_OK;
}

int hwt_surr_predict(hwt_surrogate *s, const hwt_options_f64 *o, const hwt_yield_f64 *y, double *mean, double *spread,
                     int8_t *in_box)
{
    if (!s || !valid_opts(o) || !valid_yield(y) || (o->n > 0 && (!mean || !spread || !in_box)))
        return fail(HWT_EINVAL, "hwt_surr_predict: null or negative-size argument");
    if (o->n == 0) return HWT_OK;
    DeviceGuardS dg(s->device);
    InferArgs g{};
    g.o = sopts(*o);
    g.y = SYield{y->n, y->rate, y->day};
    g.net = s->net;
    g.members = s->members;
    g.threshold = s->cfg.spread_threshold;
    g.mean = mean;
    g.spread = spread;
    g.in_box = in_box;
    k_infer<<<(o->n + INF_ROWS - 1) / INF_ROWS, 256, 0, s->stream>>>(g);
    SURR_HIP(hipGetLastError());
    SURR_HIP(hipStreamSynchronize(s->stream));
    return HWT_OK;
}

// One pricing pass, enqueued on st (for capture): the box split, the ensemble
// on the in-box rows, then the whole fallback list on the FP64 tree in one
// pass and its prices back to input order.  e1 marks the end of inference.
static int enqueue_pass(hwt_surrogate *s, hwt_plan *tree, const hwt_options_f64 *o, const hwt_yield_f64 *y,
                        double *out, hipStream_t st)
{
    uint64_t *stamps = reinterpret_cast<uint64_t *>(s->fb_count + 8);
    k_begin_pass<<<1, 64, 0, st>>>(s->fb_count, stamps);
    if (o->n == 0) {
        SURR_HIP(hipGetLastError());
        return HWT_OK;
    }
    const int blocks = (o->n + 255) / 256;
    // split: out-of-box options to the fallback list, in-box ones to the
    // inference rows (running the tree on the out-of-box part beside the
    // inference was measured slower: both compete for the same CUs)
    k_box<<<(o->n + BOX_CHUNK - 1) / BOX_CHUNK, BOX_THREADS, 0, st>>>(sopts(*o), s->fb_idx, s->fb_count, s->inf_rows,
                                                            s->fb_count + 4);
    // the ensemble on the in-box rows; options it is unsure of join the list
    InferArgs g{};
    g.o = sopts(*o);
    g.y = SYield{y->n, y->rate, y->day};
    g.net = s->net;
    g.members = s->members;
    g.threshold = s->cfg.spread_threshold;
    g.out = out;
    g.fb_idx = s->fb_idx;
    g.fb_count = s->fb_count;
    g.rows = s->inf_rows;
    g.row_count = s->fb_count + 4;
    k_infer<<<(o->n + INF_ROWS - 1) / INF_ROWS, 256, 0, st>>>(g);
    SURR_HIP(hipGetLastError());
    // the whole list on the FP64 tree in one pass
    k_fb_gather<<<blocks, 256, 0, st>>>(sopts(*o), s->fb_idx, s->fb_count, s->comp, stamps);
    const hwt_options_f64 co{o->n,          s->comp.strike, s->comp.maturity, s->comp.length, s->comp.tu,
                             s->comp.steps, s->comp.a,      s->comp.sigma,    s->comp.type};
    const int rc = hwt_internal_plan_enqueue_counted(tree, &co, s->fb_count, y, s->fb_tmp, st);
    if (rc) return rc;
    k_fb_scatter<<<blocks, 256, 0, st>>>(s->fb_idx, s->fb_count, s->fb_tmp, out, stamps);
    SURR_HIP(hipGetLastError());
    return HWT_OK;
}

int hwt_surr_price(hwt_surrogate *s, hwt_plan *tree, const hwt_options_f64 *o, const hwt_yield_f64 *y, double *out,
                   hwt_surr_stats *stats)
{
    if (!s || !tree || !valid_opts(o) || !valid_yield(y) || (o->n > 0 && !out))
        return fail(HWT_EINVAL, "hwt_surr_price: null or negative-size argument");
    if (o->n > s->infer_cap) return fail(HWT_ENOMEM, "hwt_surr_price: more options than the capacity");
    if (y->n > s->ycap) return fail(HWT_ENOMEM, "hwt_surr_price: yield curve longer than the capacity");
    // one member has no spread (always 0): a finite threshold would accept
    // every in-box price with no error estimate at all
    if (s->members < 2 && std::isfinite(s->cfg.spread_threshold))
        return fail(HWT_EINVAL, "hwt_surr_price: a one-member ensemble has no spread to gate on; "
                                "set spread_threshold to +inf to take every in-box price from the network");
    DeviceGuardS dg(s->device);
    hipStream_t st = s->stream;
    // The whole pass -- box split, ensemble inference and gate, and the FP64
    // tree on the fallback list -- is one graph, captured on the first call
    // and again when its arguments change, then replayed.
    hwt_surrogate::PassKey key;
    std::memset(&key, 0, sizeof(key));  // padding too: the key is compared bytewise
    key.o = *o;
    key.y = *y;
    key.out = out;
    key.tree = tree;
    key.tree_serial = hwt_internal_plan_serial(tree);
    key.threshold = s->cfg.spread_threshold;
    key.members = s->members;
    if (!s->exec || std::memcmp(&key, &s->key, sizeof(key)) != 0) {
        if (s->exec) (void)hipGraphExecDestroy(s->exec);
        if (s->graph) (void)hipGraphDestroy(s->graph);
        s->exec = nullptr;
        s->graph = nullptr;
        (void)hipGetLastError();
        SURR_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
        const int rc = enqueue_pass(s, tree, o, y, out, st);
        hipGraph_t g = nullptr;
        const hipError_t ec = hipStreamEndCapture(st, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (ec != hipSuccess) return fail(HWT_EHIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(ec));
        s->graph = g;
        SURR_HIP(hipGraphInstantiate(&s->exec, g, nullptr, nullptr, 0));
        s->key = key;
    }
    SURR_HIP(hipEventRecord(s->e0, st));
    SURR_HIP(hipGraphLaunch(s->exec, st));
    if (o->n > 0) hwt_internal_plan_replayed_on(tree, st);
    SURR_HIP(hipEventRecord(s->e2, st));
    SURR_HIP(hipMemcpyAsync(s->h_count, s->fb_count, 16 * sizeof(int32_t), hipMemcpyDeviceToHost, st));
    SURR_HIP(hipStreamSynchronize(st));
    const int trc = o->n > 0 ? hwt_plan_sync(tree, nullptr) : HWT_OK;
    if (stats) {
        std::memset(stats, 0, sizeof(*stats));
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, s->e0, s->e2) == hipSuccess) stats->ms = ms;
        uint64_t t[3];
        std::memcpy(t, s->h_count + 8, sizeof(t));
        stats->surrogate_ms = (double)(t[1] - t[0]) / s->wall_khz;
        stats->tree_ms = (double)(t[2] - t[1]) / s->wall_khz;
        stats->fallback = s->h_count[0];
        stats->out_of_box = s->h_count[1];
        stats->steps = s->step;
    }
    return trc;
}

int hwt_surr_save(hwt_surrogate *s, const char *path)
{
    if (!s || !path) return fail(HWT_EINVAL, "hwt_surr_save: bad arguments");
    DeviceGuardS dg(s->device);
    const size_t nm = (size_t)s->members * PSTRIDE;
    std::vector<float> P(nm), m1(nm), m2(nm);
    SURR_HIP(hipStreamSynchronize(s->stream));
    SURR_HIP(hipMemcpy(P.data(), s->net.P, nm * 4, hipMemcpyDeviceToHost));
    SURR_HIP(hipMemcpy(m1.data(), s->m1, nm * 4, hipMemcpyDeviceToHost));
    SURR_HIP(hipMemcpy(m2.data(), s->m2, nm * 4, hipMemcpyDeviceToHost));
    std::ostringstream rs;
    rs << s->rng;
    const std::string rng = rs.str();
    FILE *f = std::fopen(path, "wb");
    if (!f) return fail(HWT_EINVAL, std::string("hwt_surr_save: cannot open ") + path);
    const char magic[8] = {'H', 'W', 'T', 'S', 'U', 'R', 'R', '1'};
    const int32_t hdr[4] = {s->members, NPAR, PSTRIDE, s->epochs_done};
    const int64_t step = s->step, rl = (int64_t)rng.size();
    bool ok = std::fwrite(magic, 1, 8, f) == 8 && std::fwrite(hdr, 4, 4, f) == 4 && std::fwrite(&step, 8, 1, f) == 1 &&
              std::fwrite(&rl, 8, 1, f) == 1 && std::fwrite(rng.data(), 1, rng.size(), f) == rng.size() &&
              std::fwrite(P.data(), 4, nm, f) == nm && std::fwrite(m1.data(), 4, nm, f) == nm &&
              std::fwrite(m2.data(), 4, nm, f) == nm;
    ok = (std::fclose(f) == 0) && ok;
    return ok ? HWT_OK : fail(HWT_EINVAL, std::string("hwt_surr_save: write failed: ") + path);
}

int hwt_surr_load(hwt_surrogate *s, const char *path)
{
    if (!s || !path) return fail(HWT_EINVAL, "hwt_surr_load: bad arguments");
    DeviceGuardS dg(s->device);
    FILE *f = std::fopen(path, "rb");
    if (!f) return fail(HWT_EINVAL, std::string("hwt_surr_load: cannot open ") + path);
    char magic[8];
    int32_t hdr[4];
    int64_t step = 0, rl = 0;
    bool ok = std::fread(magic, 1, 8, f) == 8 && std::memcmp(magic, "HWTSURR1", 8) == 0 &&
              std::fread(hdr, 4, 4, f) == 4 && hdr[0] == s->members && hdr[1] == NPAR && hdr[2] == PSTRIDE &&
              std::fread(&step, 8, 1, f) == 1 && std::fread(&rl, 8, 1, f) == 1 && rl > 0 && rl < (1 << 20);
    std::string rng;
    const size_t nm = (size_t)s->members * PSTRIDE;
    std::vector<float> P(nm), m1(nm), m2(nm);
    if (ok) {
        rng.resize((size_t)rl);
        ok = std::fread(&rng[0], 1, rng.size(), f) == rng.size() && std::fread(P.data(), 4, nm, f) == nm &&
             std::fread(m1.data(), 4, nm, f) == nm && std::fread(m2.data(), 4, nm, f) == nm;
    }
    std::fclose(f);
    if (!ok) return fail(HWT_EINVAL, std::string("hwt_surr_load: not a compatible checkpoint: ") + path);
    std::istringstream is(rng);
    is >> s->rng;
    s->step = step;
    s->epochs_done = hdr[3];
    SURR_HIP(hipStreamSynchronize(s->stream));
    SURR_HIP(hipMemcpy(s->net.P, P.data(), nm * 4, hipMemcpyHostToDevice));
    SURR_HIP(hipMemcpy(s->m1, m1.data(), nm * 4, hipMemcpyHostToDevice));
    SURR_HIP(hipMemcpy(s->m2, m2.data(), nm * 4, hipMemcpyHostToDevice));
    k_refresh_bf16<<<dim3((3 * LAYER_W + 255) / 256, s->members), 256, 0, s->stream>>>(s->net, s->members);
    SURR_HIP(hipGetLastError());
    SURR_HIP(hipStreamSynchronize(s->stream));
    return HWT_OK;
}

} // extern "C"
