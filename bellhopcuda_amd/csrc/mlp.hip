// mlp.hip -- the TL surrogate's network: an MLP ensemble trained on tracer
// fields, forward and backward on gfx950 matrix cores (BF16 inputs, FP32
// accumulate).
//
// Network (one ensemble member; E members are trained side by side):
//   16 normalised inputs -> 64 features -> 6 hidden layers of 256 units, GELU
//   (erf form) -> n_out outputs (linear). Features: front 0, [sin, cos](2 pi B x)
//   of 32 projections B x; front 1, the 16 inputs themselves followed by
//   [sin, cos] of the first 24 projections. n_out = 1 gives a coordinate
//   network (TL at one receiver); n_out = K (a multiple of 32, <= 256) gives
//   the K coefficients of a field expanded in a fixed basis. Weights are kept
//   in FP32 (master, Adam state) and as a BF16 copy that the matrix products
//   read; hidden activations are stored in BF16, the GELU's slopes in FP32.
//
// The rows of a batch are independent through the whole network, so k_rows
// takes 32 of them from the inputs to the outputs and, in training, back to the
// first layer's gradient in one launch: activations pass from layer to layer in
// LDS, weights are read from the L2 in the matrix cores' operand order, and
// only the GELU's slopes go to memory, FP32, for the thread that made them.
// What the weight gradients need (activations and layer gradients, BF16) is
// written in operand order too, so that k_wgrad reads both operands of H^T dZ
// straight into registers. A training step is k_rows, k_wgrad and k_adam.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/bhc_hip.h"

// hipMalloc that gives idle blocks of the library's contexts back before it gives up
hipError_t bhc_device_malloc(void **p, size_t n);

namespace {

thread_local std::string g_mlp_error;
int mfail(const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_mlp_error = buf;
    return -1;
}
#define MCHECK(x) \
    do { \
        hipError_t _e = (x); \
        if(_e != hipSuccess) return mfail("%s failed: %s (%s:%d)", #x, hipGetErrorString(_e), __FILE__, __LINE__); \
    } while(0)

constexpr int D_IN = 16, N_FREQ = 32, D_FF = 2 * N_FREQ, WIDTH = 256, N_HID = 6;
constexpr int N_FREQ_RAW = (D_FF - D_IN) / 2; // projections used by front 1
constexpr int ROWS = 32;           // batch rows per workgroup of k_rows
constexpr int NT_W = WIDTH / 32;   // 32-column tiles of a hidden layer

typedef uint16_t bf16_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// parameter layout of one member (floats): W0 [D_FF][WIDTH], b0 [WIDTH],
// W1..W5 [WIDTH][WIDTH], b1..b5 [WIDTH], Wout [WIDTH][n_out], bout [n_out]
constexpr size_t off_W(int l) { return l == 0 ? 0 : (size_t)(D_FF + 1) * WIDTH + (size_t)(l - 1) * (WIDTH + 1) * WIDTH; }
constexpr size_t off_b(int l) { return off_W(l) + (size_t)(l == 0 ? D_FF : WIDTH) * WIDTH; }
constexpr size_t OFF_WOUT = off_W(N_HID);
constexpr size_t off_bout(int n_out) { return OFF_WOUT + (size_t)WIDTH * n_out; }
constexpr size_t n_param(int n_out) { return off_bout(n_out) + n_out; }

__host__ __device__ inline bf16_t f2bf(float f)
{ // round to nearest even
    uint32_t u;
    memcpy(&u, &f, 4);
    if((u & 0x7F800000u) == 0x7F800000u) return (bf16_t)(u >> 16); // inf / nan
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(bf16_t h)
{
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}
// The same rounding by the hardware's conversion (one instruction for two values).
__device__ inline bf16_t cvt_bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }
// GELU (erf form) of z from c = 1 + erf(z / sqrt 2), and its derivative.
__device__ inline float gelu_c(float z) { return 1.0f + erff(z * 0.70710678118654752f); }
__device__ inline float gelu(float z, float c) { return 0.5f * z * c; }
__device__ inline float gelu_d(float z, float c) { return 0.5f * c + z * 0.39894228040143268f * expf(-0.5f * z * z); }

// Operand order of a K x N matrix: blocks of 16 K values by 32 columns, K-major,
// NT = N / 32 blocks across; a block holds 64 lanes' 8 values, lane l those of
// column l % 32 at K = 8 (l / 32) .. + 7 (v_mfma_f32_32x32x16_bf16's A and B).
__host__ __device__ inline size_t op_at(int k, int n, int NT)
{
    return (((size_t)(k >> 4) * NT + (n >> 5)) * 64 + (n & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
}

struct RowArgs {
    const float *X, *Y;        // inputs [.][16] and targets [.][n_out]; row b of the batch is idx[b] (b without idx)
    const int32_t *idx;
    int n, n_out, front;
    const float *Bf;           // [N_FREQ][D_IN]
    const bf16_t *Wf, *Wb;     // weights in operand order, for the forward and the backward products
    const float *P;            // FP32 parameters (biases)
    long long np, npf;         // parameters and BF16 copy's elements per member
    float *out;                // [members][n][n_out] (prediction)
    bf16_t *F;                 // operand order over the batch rows: features,
    bf16_t *H[N_HID], *dZ[N_HID], *dO; // activations, layer gradients and output gradient [member]
    long long zH, zO;          // elements per member of H / dZ and of dO
    float *D[N_HID];           // GELU'(Z) [member][row block][16][512]: each thread's own values
    int members;
    float *G, *loss;
};

typedef __attribute__((__vector_size__(4 * sizeof(uint16_t)))) uint16_t u16x4;

// The weights of one 32 x 32 product: column block nt of W (operand order, KT
// blocks deep), and the product of the rows of act (LDS) with them.
template<int KT> __device__ inline void load_w(bf16x8 *b, const bf16_t *W, int NT, int nt, int lane)
{
#pragma unroll
    for(int kt = 0; kt < KT; ++kt)
        b[kt] = *reinterpret_cast<const bf16x8 *>(W + (((size_t)kt * NT + nt) * 64 + lane) * 8);
}
template<int KT> __device__ inline f32x16 row_product(const bf16_t (*act)[WIDTH + 8], const bf16x8 *b, int lane)
{
    f32x16 acc = {};
#pragma unroll
    for(int kt = 0; kt < KT; ++kt) {
        bf16x8 a = *reinterpret_cast<const bf16x8 *>(&act[lane & 31][kt * 16 + 8 * (lane >> 5)]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[kt], acc, 0, 0, 0);
    }
    return acc;
}

// Row of accumulator register r in a 32 x 32 product (column: lane % 32).
__device__ inline int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// The 16 values of a lane's column as BF16: rows of the next product's
// activations in LDS (act, if given) and operand order over the batch rows
// (op, if given: block row rb * 2, nt of NT).
__device__ inline void put_cols(const float *v, bf16_t (*act)[WIDTH + 8], bf16_t *op, int rb, int NT, int nt, int lane)
{
#pragma unroll
    for(int g = 0; g < 4; ++g) {
        u16x4 q;
#pragma unroll
        for(int i = 0; i < 4; ++i) {
            q[i] = cvt_bf(v[4 * g + i]);
            if(act) act[acc_row(4 * g + i, lane)][nt * 32 + (lane & 31)] = q[i];
        }
        if(op)
            *reinterpret_cast<u16x4 *>(op + (((size_t)(rb * 2 + (g >> 1)) * NT + nt) * 64 + (lane & 31) + 32 * (g & 1)) * 8
                                       + 4 * (lane >> 5)) = q;
    }
}

// Sum of a lane's column over the 32 rows, added to *to once per column.
__device__ inline void add_col(const float *v, float *to, int lane)
{
    float s = 0.f;
#pragma unroll
    for(int r = 0; r < 16; ++r) s += v[r];
    s += __shfl_xor(s, 32);
    if(lane < 32) unsafeAtomicAdd(to, s);
}

// ROWS batch rows of one member through the network, and in training (TRAIN)
// the loss, the output gradient and every layer's gradient dZ back to the
// first layer. Eight wavefronts, one 32-column tile of each layer apiece: two
// per SIMD. 2048 rows of 4 members are 256 workgroups, one per CU. Waiting bounds
// it: a wavefront waits for memory or a layer's barrier in 62 % of its cycles and
// issues vector instructions in 16 % (12.6 million GELUs a step of some 65
// instructions, made once: the slope is kept, not the pre-activation), and two
// wavefronts per SIMD cannot cover that. In its 86 us it writes 105 MB (half of
// it slopes) and reads 99, and the L2 answers 5.1 million requests, the weights'
// above all. A layer's weights (128 KB per workgroup, from the L2) are loaded
// while the layer before goes through its GELU.
// Replaces one launch per layer and direction with FP32 pre-activations and
// gradients in memory: a training step of 2048 rows, 4 members, 128 outputs
// took 1270 us in 36 launches (28 us of it at the matrix cores' rate).
template<bool TRAIN> __global__ void __launch_bounds__(512) k_rows(RowArgs g)
{
    __shared__ __align__(16) bf16_t act[2][ROWS][WIDTH + 8];
    __shared__ float grow[ROWS];   // single output: its gradient per row
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int rb = blockIdx.x, e = blockIdx.y, r0 = rb * ROWS;
    const float *P = g.P + e * g.np;
    const bf16_t *Wf = g.Wf + e * g.npf, *Wb = g.Wb + e * g.npf;
    float *G = TRAIN ? g.G + e * g.np : nullptr;
    const int col = wave * 32 + (lane & 31);
    // features of normalised inputs. Front 0: F[2j] = sin(2 pi <B_j, x>),
    // F[2j + 1] = cos, j < 32. Front 1: F[d] = x[d], d < 16, then sin / cos of
    // projections j < 24 at F[16 + 2j], F[17 + 2j].
    for(int i = t; i < ROWS * N_FREQ; i += 512) {
        const int row = i / N_FREQ, j = i % N_FREQ, b = r0 + row;
        float v0 = 0.f, v1 = 0.f;
        int o = 2 * j;
        if(g.front == 1) o = j >= N_FREQ_RAW ? 2 * (j - N_FREQ_RAW) : D_IN + 2 * j;
        if(b < g.n) {
            const float *x = g.X + (size_t)(g.idx ? g.idx[b] : b) * D_IN;
            if(g.front == 1 && j >= N_FREQ_RAW) {
                v0 = x[o];
                v1 = x[o + 1];
            } else {
                float s = 0.f;
                for(int d = 0; d < D_IN; ++d) s += g.Bf[j * D_IN + d] * x[d];
                sincospif(2.0f * s, &v0, &v1);
            }
        }
        act[0][row][o] = f2bf(v0);
        act[0][row][o + 1] = f2bf(v1);
    }
    __syncthreads();
    if(TRAIN && e == 0 && t < 256) { // features in operand order over the rows
        const int kt = t >> 7, nt = (t >> 6) & 1, c = nt * 32 + (lane & 31), k0 = kt * 16 + 8 * (lane >> 5);
        alignas(16) bf16_t q[8];
        for(int j = 0; j < 8; ++j) q[j] = act[0][k0 + j][c];
        *reinterpret_cast<uint4 *>(g.F + (((size_t)(rb * 2 + kt) * 2 + nt) * 64 + lane) * 8) = *reinterpret_cast<uint4 *>(q);
    }
    // GELU' (FP32) of this lane's column, kept for the way back
    const size_t ds = ((size_t)e * gridDim.x + rb) * 16 * 512 + t;
    int cur = 0;
    bf16x8 w[WIDTH / 16];
    load_w<D_FF / 16>(w, Wf, NT_W, wave, lane);
#pragma unroll 1
    for(int l = 0; l < N_HID; ++l) {
        const f32x16 acc = l == 0 ? row_product<D_FF / 16>(act[cur], w, lane) : row_product<WIDTH / 16>(act[cur], w, lane);
        const float bias = P[off_b(l) + col];
        if(l + 1 < N_HID) load_w<WIDTH / 16>(w, Wf + off_W(l + 1), NT_W, wave, lane);
        float h[16];
#pragma unroll
        for(int r = 0; r < 16; ++r) {
            const float z = acc[r] + bias, c = gelu_c(z);
            if(TRAIN) g.D[l][ds + r * 512] = gelu_d(z, c);
            h[r] = gelu(z, c);
        }
        put_cols(h, act[cur ^ 1], TRAIN ? g.H[l] + e * g.zH : nullptr, rb, NT_W, wave, lane);
        cur ^= 1;
        __syncthreads();
    }
    // output layer, and in training the loss and its gradient
    float lsum = 0.f;
    const float total = (float)(g.n * g.n_out);
    if(g.n_out == 1) {
        for(int k = 0; k < 4; ++k) {
            const int row = wave * 4 + k;
            float s = 0.f;
            for(int j = 0; j < 4; ++j) s += bf2f(act[cur][row][lane * 4 + j]) * bf2f(Wf[OFF_WOUT + lane * 4 + j]);
            for(int o = 32; o; o >>= 1) s += __shfl_xor(s, o);
            s += P[off_bout(1)];
            const int b = r0 + row;
            if(lane == 0 && b < g.n) {
                if(TRAIN) {
                    const float d = s - g.Y[g.idx ? g.idx[b] : b];
                    grow[row] = 2.0f * d / total;
                    lsum += d * d / total;
                } else {
                    g.out[(size_t)e * g.n + b] = s;
                }
            }
        }
        if(!TRAIN) return;
        __syncthreads();
        if(t < WIDTH) {
            float s = 0.f;
            for(int r = 0; r < ROWS; ++r) s += bf2f(act[cur][r][t]) * grow[r];
            unsafeAtomicAdd(G + OFF_WOUT + t, s);
        } else if(t == WIDTH) {
            float s = 0.f;
            for(int r = 0; r < ROWS; ++r) s += grow[r];
            unsafeAtomicAdd(G + off_bout(1), s);
        }
    } else {
        const int NT = g.n_out / 32;
        if(wave < NT) {
            load_w<WIDTH / 16>(w, Wf + OFF_WOUT, NT, wave, lane);
            const f32x16 acc = row_product<WIDTH / 16>(act[cur], w, lane);
            const float bias = P[off_bout(g.n_out) + col];
            float d[16];
#pragma unroll
            for(int r = 0; r < 16; ++r) {
                const int b = r0 + acc_row(r, lane);
                const float v = acc[r] + bias;
                d[r] = 0.f;
                if(b < g.n) {
                    if(TRAIN) {
                        const float df = v - g.Y[(size_t)(g.idx ? g.idx[b] : b) * g.n_out + col];
                        lsum += df * df / total;
                        d[r] = 2.0f * df / total;
                    } else {
                        g.out[((size_t)e * g.n + b) * g.n_out + col] = v;
                    }
                }
            }
            if(TRAIN) {
                add_col(d, G + off_bout(g.n_out) + col, lane);
                put_cols(d, act[cur ^ 1], g.dO + (size_t)e * g.zO, rb, NT, wave, lane);
            }
        }
        if(!TRAIN) return;
        cur ^= 1;
        __syncthreads();
    }
    for(int o = 32; o; o >>= 1) lsum += __shfl_xor(lsum, o);
    if(lane == 0) unsafeAtomicAdd(g.loss + e, lsum);
    // back through the layers: dZ_l = (dZ_{l+1} W_{l+1}^T) GELU'(Z_l)
#pragma unroll 1
    for(int l = N_HID - 1; l >= 0; --l) {
        float d[16], slope[16];
#pragma unroll
        for(int r = 0; r < 16; ++r) slope[r] = g.D[l][ds + r * 512];
        if(l == N_HID - 1 && g.n_out == 1) {
            const float wo = bf2f(Wf[OFF_WOUT + col]);
#pragma unroll
            for(int r = 0; r < 16; ++r) d[r] = grow[acc_row(r, lane)] * wo;
        } else {
            f32x16 acc = {};
            if(l == N_HID - 1) {
                const bf16_t *W = Wb + OFF_WOUT;
                for(int kt = 0; kt < g.n_out / 16; ++kt) {
                    bf16x8 b = *reinterpret_cast<const bf16x8 *>(W + (((size_t)kt * NT_W + wave) * 64 + lane) * 8);
                    bf16x8 a = *reinterpret_cast<const bf16x8 *>(&act[cur][lane & 31][kt * 16 + 8 * (lane >> 5)]);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
                }
            } else {
                acc = row_product<WIDTH / 16>(act[cur], w, lane);
            }
#pragma unroll
            for(int r = 0; r < 16; ++r) d[r] = acc[r];
        }
        if(l > 0) load_w<WIDTH / 16>(w, Wb + off_W(l), NT_W, wave, lane);
#pragma unroll
        for(int r = 0; r < 16; ++r) d[r] *= slope[r];
        add_col(d, G + off_b(l) + col, lane);
        put_cols(d, l > 0 ? act[cur ^ 1] : nullptr, g.dZ[l] + e * g.zH, rb, NT_W, wave, lane);
        cur ^= 1;
        __syncthreads();
    }
}

// Weight gradients dW = H^T dZ of every layer and member: one workgroup per
// 64 x 32 tile, its four wavefronts splitting the batch rows; both operands
// come in operand order, 16 bytes per lane, and the four partial tiles are
// summed in LDS in a fixed order. A layer's tiles read the same two matrices
// (2 MB at 2048 rows), so the workgroups of one (layer, member) are dealt to
// one XCD (workgroups go to the eight XCDs in turn) and share its L2.
constexpr int WG_TILES = (WIDTH / 64) * NT_W;
__global__ void __launch_bounds__(256) k_wgrad(RowArgs g)
{
    const int n = g.n, n_out = g.n_out, members = g.members;
    __shared__ float part[4][64 * 32];
    const int nlayer = n_out > 1 ? N_HID + 1 : N_HID;
    const int q = blockIdx.x >> 3, combo = (blockIdx.x & 7) + 8 * (q / WG_TILES), tile = q % WG_TILES;
    if(combo >= nlayer * members) return;
    const int l = combo % nlayer, e = combo / nlayer;
    const int Kin = l == 0 ? D_FF : WIDTH, N = l == N_HID ? n_out : WIDTH;
    const int NTa = Kin / 32, NTb = N / 32;
    const int mp = tile / NTb, nt = tile % NTb;
    if(mp >= Kin / 64) return;
    const bf16_t *A = l == 0 ? g.F : g.H[l - 1] + e * g.zH;
    const bf16_t *B = l == N_HID ? g.dO + e * g.zO : g.dZ[l] + e * g.zH;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int nk = n / 16, k0 = wave * nk / 4, k1 = (wave + 1) * nk / 4;
    f32x16 c0 = {}, c1 = {};
    for(int kt = k0; kt < k1; ++kt) {
        const bf16_t *a = A + (((size_t)kt * NTa + 2 * mp) * 64 + lane) * 8;
        bf16x8 a0 = *reinterpret_cast<const bf16x8 *>(a), a1 = *reinterpret_cast<const bf16x8 *>(a + 512);
        bf16x8 b = *reinterpret_cast<const bf16x8 *>(B + (((size_t)kt * NTb + nt) * 64 + lane) * 8);
        c0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b, c0, 0, 0, 0);
        c1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b, c1, 0, 0, 0);
    }
    for(int r = 0; r < 16; ++r) {
        part[wave][acc_row(r, lane) * 32 + (lane & 31)] = c0[r];
        part[wave][(32 + acc_row(r, lane)) * 32 + (lane & 31)] = c1[r];
    }
    __syncthreads();
    float *W = g.G + e * g.np + off_W(l);
    for(int i = t; i < 64 * 32; i += 256)
        W[(size_t)(mp * 64 + (i >> 5)) * N + nt * 32 + (i & 31)] = part[0][i] + part[1][i] + part[2][i] + part[3][i];
}

// Weight tiles of 32 x 32 in a member, layer by layer, K-major within a layer
// (the output layer's only with several outputs).
__host__ __device__ inline int n_tiles(int n_out)
{
    return (D_FF / 32 + (N_HID - 1) * NT_W) * NT_W + (n_out > 1 ? NT_W * (n_out / 32) : 0);
}
struct WTile {
    size_t W;                  // the layer's first weight
    int N, k0, n0, layer;
};
__device__ inline WTile w_tile(int q, int n_out)
{
    WTile t;
    const int first = (D_FF / 32) * NT_W;
    if(q < first) t.layer = 0;
    else {
        q -= first;
        t.layer = 1 + min(q / (NT_W * NT_W), N_HID - 1);
        q -= (t.layer - 1) * NT_W * NT_W;
    }
    t.W = off_W(t.layer);
    t.N = t.layer == N_HID ? n_out : WIDTH;
    t.k0 = q / (t.N / 32) * 32;
    t.n0 = q % (t.N / 32) * 32;
    return t;
}

// The BF16 copies of a tile (tile[k][n], by the 256 threads of a workgroup) in
// operand order for both directions, 16 bytes per thread.
__device__ inline void put_tile(const bf16_t (*tile)[34], const WTile &w, bf16_t *Wf, bf16_t *Wb)
{
    const int t = threadIdx.x & 127, kt = t >> 6, lane = t & 63, c = lane & 31, r0 = kt * 16 + 8 * (lane >> 5);
    alignas(16) bf16_t q[8];
    if(threadIdx.x < 128) { // K = row, N = column
        for(int j = 0; j < 8; ++j) q[j] = tile[r0 + j][c];
        *reinterpret_cast<uint4 *>(Wf + w.W + op_at(w.k0 + r0, w.n0 + c, w.N / 32)) = *reinterpret_cast<uint4 *>(q);
    } else if(w.layer > 0) { // K = column, N = row
        for(int j = 0; j < 8; ++j) q[j] = tile[c][r0 + j];
        *reinterpret_cast<uint4 *>(Wb + w.W + op_at(w.n0 + r0, w.k0 + c, NT_W)) = *reinterpret_cast<uint4 *>(q);
    }
}

// Parameter number j of those that are no tile's: the biases layer by layer,
// then a single output's weights; -1 past the last.
__device__ inline long long loose_param(int j, int n_out)
{
    if(j < N_HID * WIDTH) return (long long)off_b(j / WIDTH) + j % WIDTH;
    j -= N_HID * WIDTH;
    if(j < n_out) return (long long)off_bout(n_out) + j;
    j -= n_out;
    return n_out == 1 && j < WIDTH ? (long long)OFF_WOUT + j : -1;
}
__host__ __device__ inline int n_loose(int n_out) { return N_HID * WIDTH + n_out + (n_out == 1 ? WIDTH : 0); }

__global__ void k_zero(float *p, long long n)
{
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if(i < n) p[i] = 0.0f;
}

// Adam (FP32 master weights), the BF16 copies the products read, and zeros for
// the next step's loss and for the gradients that k_rows adds to (biases, a
// single output's weights). One workgroup per 32 x 32 tile of weights, which
// goes through LDS so that both copies are stored 16 bytes at a time; the last
// workgroups take the loose parameters. Member: blockIdx.y. STEP = false only
// makes the copies.
template<bool STEP>
__global__ void __launch_bounds__(256) k_adam(float *Pm, float *M, float *V, float *Gm, bf16_t *Wf, bf16_t *Wb, long long np,
                                              long long npf, int n_out, float lr, float b1, float b2, float eps, float c1,
                                              float c2, float *next_loss)
{
    __shared__ bf16_t tile[32][34];
    const int e = blockIdx.y, t = threadIdx.x, nt = n_tiles(n_out);
    float *P = Pm + e * np, *G = STEP ? Gm + e * np : nullptr;
    Wf += e * npf;
    Wb += e * npf;
    auto step = [&](size_t i) {
        float p = P[i];
        if(STEP) {
            const size_t s = e * np + i;
            const float g = G[i];
            const float m = b1 * M[s] + (1.0f - b1) * g;
            const float v = b2 * V[s] + (1.0f - b2) * g * g;
            M[s] = m;
            V[s] = v;
            p = p - lr * (m / c1) / (sqrtf(v / c2) + eps);
            P[i] = p;
        }
        return p;
    };
    if((int)blockIdx.x < nt) {
        const WTile w = w_tile((int)blockIdx.x, n_out);
        for(int r = t >> 5; r < 32; r += 8) tile[r][t & 31] = cvt_bf(step(w.W + (size_t)(w.k0 + r) * w.N + w.n0 + (t & 31)));
        __syncthreads();
        put_tile(tile, w, Wf, Wb);
        return;
    }
    const int j = ((int)blockIdx.x - nt) * 256 + t;
    if(STEP && j == 0) next_loss[e] = 0.f;
    const long long i = loose_param(j, n_out);
    if(i < 0) return;
    const float p = step((size_t)i);
    if(STEP) G[i] = 0.f;
    if(n_out == 1 && i >= (long long)OFF_WOUT && i < (long long)off_bout(1)) Wf[i] = cvt_bf(p);
}

} // namespace

struct bhc_mlp {
    int device;
    hipStream_t stream;
    int members, max_batch;
    int n_out, front;          // outputs per point; feature front (0 Fourier, 1 inputs + Fourier)
    long long np, npf;         // parameters per member; elements per member of a BF16 copy
    float *P, *Mo, *Vo, *G;    // [members][np]
    bf16_t *Wf, *Wb;           // [members][npf]: weights in operand order, forward and backward
    float *Bf;                 // [N_FREQ][D_IN]
    float *x, *y, *out, *loss; // x [max_batch][16], y [max_batch][n_out], out [members][max_batch][n_out], loss [2][16]
    bf16_t *F;                 // features [max_batch][D_FF], operand order over the rows
    bf16_t *H[N_HID], *dZ[N_HID]; // [members][max_batch][WIDTH], operand order over the rows
    bf16_t *dO;                // [members][max_batch][n_out], operand order over the rows
    float *D[N_HID];           // GELU'(Z) [members][max_batch / 32][16][512]
    float *X, *Y;              // resident training set: X [nset][16], Y [nset][n_out]
    int32_t *idx;              // batches of a chunk of steps
    long long nset;
    long long step;
    int last_loss;             // which half of `loss` holds the last step's
    hipEvent_t e0, e1;
    double last_ms;
};

namespace {

constexpr int IDX_CHUNK = 8;   // training steps whose batches are drawn and copied at a time

RowArgs row_args(bhc_mlp *m, const float *X, const float *Y, const int32_t *idx, int n, float *loss)
{
    RowArgs g;
    g.X = X;
    g.Y = Y;
    g.idx = idx;
    g.n = n;
    g.n_out = m->n_out;
    g.front = m->front;
    g.Bf = m->Bf;
    g.Wf = m->Wf;
    g.Wb = m->Wb;
    g.P = m->P;
    g.np = m->np;
    g.npf = m->npf;
    g.out = m->out;
    g.F = m->F;
    for(int l = 0; l < N_HID; ++l) {
        g.H[l] = m->H[l];
        g.dZ[l] = m->dZ[l];
        g.D[l] = m->D[l];
    }
    g.dO = m->dO;
    g.zH = (long long)m->max_batch * WIDTH;
    g.zO = (long long)m->max_batch * m->n_out;
    g.members = m->members;
    g.G = m->G;
    g.loss = loss;
    return g;
}

// forward of n points X [n][16]: out [members][n][n_out]
void forward(bhc_mlp *m, const float *X, int n)
{
    hipLaunchKernelGGL(k_rows<false>, dim3((n + ROWS - 1) / ROWS, m->members), dim3(512), 0, m->stream,
                       row_args(m, X, nullptr, nullptr, n, nullptr));
}

// forward and backward of a batch of n rows (a multiple of 32): gradients in
// m->G (whose added slots are zero before), loss added to `loss`
void forward_backward(bhc_mlp *m, const float *X, const float *Y, const int32_t *idx, int n, float *loss)
{
    const RowArgs g = row_args(m, X, Y, idx, n, loss);
    hipLaunchKernelGGL(k_rows<true>, dim3(n / ROWS, m->members), dim3(512), 0, m->stream, g);
    const int combos = (m->n_out > 1 ? N_HID + 1 : N_HID) * m->members;
    hipLaunchKernelGGL(k_wgrad, dim3((unsigned)((combos + 7) / 8 * 8 * WG_TILES)), dim3(256), 0, m->stream, g);
}

void refresh_bf(bhc_mlp *m)
{
    hipLaunchKernelGGL(k_adam<false>, dim3(n_tiles(m->n_out) + (n_loose(m->n_out) + 255) / 256, m->members), dim3(256), 0,
                       m->stream, m->P, nullptr, nullptr, nullptr, m->Wf, m->Wb, m->np, m->npf, m->n_out, 0.f, 0.f, 0.f,
                       0.f, 0.f, 0.f, nullptr);
}

void zero_grads(bhc_mlp *m)
{
    const long long np = (long long)m->members * m->np;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, m->stream, m->G, np);
    hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, m->stream, m->loss, 32ll);
}

} // namespace

extern "C" const char *bhc_mlp_last_error(void) { return g_mlp_error.c_str(); }

extern "C" int bhc_mlp_num_params(void) { return (int)n_param(1); }

extern "C" long long bhc_mlp_param_count(bhc_mlp *m) { return m ? m->np : 0; }

extern "C" void bhc_mlp_destroy(bhc_mlp *m)
{
    if(!m) return;
    (void)hipSetDevice(m->device);
    (void)hipStreamSynchronize(m->stream);
    void *ptrs[] = {m->P, m->Mo, m->Vo, m->G, m->Wf, m->Wb, m->Bf, m->x, m->y, m->out, m->loss, m->F, m->dO, m->X, m->Y,
                    m->idx};
    for(void *p : ptrs)
        if(p) (void)hipFree(p);
    for(int l = 0; l < N_HID; ++l)
        for(void *p : {(void *)m->H[l], (void *)m->D[l]})
            if(p) (void)hipFree(p);
    (void)hipEventDestroy(m->e0);
    (void)hipEventDestroy(m->e1);
    (void)hipStreamDestroy(m->stream);
    delete m;
}

// Create an ensemble of `members` networks with n_out outputs (1, or a
// multiple of 32 up to 256) and feature front `front` (0 or 1), for batches of
// up to max_batch points (a multiple of 32). Weights: He-uniform from `seed`,
// biases and the output layer 0; the projection matrix has N(0, sigma^2)
// entries from the same seed.
extern "C" int bhc_mlp_create_ex(int device, int members, int max_batch, int n_out, int front,
                                 unsigned long long seed, float sigma, bhc_mlp **out)
{
    *out = nullptr;
    if(members < 1 || members > 16 || max_batch < 32 || max_batch % 32) return mfail("bhc_mlp_create: bad sizes");
    if(!(n_out == 1 || (n_out % 32 == 0 && n_out <= WIDTH))) return mfail("bhc_mlp_create: n_out must be 1 or a multiple of 32 <= 256");
    if(front != 0 && front != 1) return mfail("bhc_mlp_create: front must be 0 or 1");
    MCHECK(hipSetDevice(device));
    bhc_mlp *m = new bhc_mlp();
    memset(m, 0, sizeof(*m));
    m->device = device;
    m->members = members;
    m->max_batch = max_batch;
    m->n_out = n_out;
    m->front = front;
    m->np = (long long)n_param(n_out);
    m->npf = (m->np + 63) / 64 * 64;
    MCHECK(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking));
    MCHECK(hipEventCreate(&m->e0));
    MCHECK(hipEventCreate(&m->e1));
    size_t np = (size_t)members * m->np;
    size_t act = (size_t)members * max_batch * WIDTH;
    size_t outs = (size_t)max_batch * n_out;
    const size_t npf = (size_t)members * m->npf;
    bool bad = bhc_device_malloc((void **)&m->P, np * 4) || bhc_device_malloc((void **)&m->Mo, np * 4)
        || bhc_device_malloc((void **)&m->Vo, np * 4) || bhc_device_malloc((void **)&m->G, np * 4)
        || bhc_device_malloc((void **)&m->Wf, npf * 2) || bhc_device_malloc((void **)&m->Wb, npf * 2)
        || bhc_device_malloc((void **)&m->Bf, N_FREQ * D_IN * 4)
        || bhc_device_malloc((void **)&m->x, (size_t)max_batch * D_IN * 4) || bhc_device_malloc((void **)&m->y, outs * 4)
        || bhc_device_malloc((void **)&m->out, (size_t)members * outs * 4) || bhc_device_malloc((void **)&m->loss, 32 * 4)
        || bhc_device_malloc((void **)&m->F, (size_t)max_batch * D_FF * 2)
        || bhc_device_malloc((void **)&m->dO, (size_t)members * outs * 2)
        || bhc_device_malloc((void **)&m->idx, IDX_CHUNK * (size_t)max_batch * 4);
    for(int l = 0; l < N_HID && !bad; ++l)
        bad = bhc_device_malloc((void **)&m->H[l], act * 4) || bhc_device_malloc((void **)&m->D[l], act * 4);
    for(int l = 0; l < N_HID && !bad; ++l) m->dZ[l] = m->H[l] + act; // second half of H's block
    if(bad) {
        bhc_mlp_destroy(m);
        return mfail("bhc_mlp_create: out of device memory");
    }
    std::mt19937_64 rng(seed);
    std::vector<float> P(np, 0.0f), Bf(N_FREQ * D_IN);
    std::normal_distribution<double> nd(0.0, 1.0);
    for(auto &b : Bf) b = (float)(sigma * nd(rng));
    // hidden layers: He-uniform; the output layer starts at zero, so that a
    // network trained on residuals starts from the reference it corrects
    for(int e = 0; e < members; ++e) {
        for(int l = 0; l < N_HID; ++l) {
            int fan_in = l == 0 ? D_FF : WIDTH;
            double a = std::sqrt(6.0 / fan_in);
            std::uniform_real_distribution<double> ud(-a, a);
            size_t o = (size_t)e * m->np + off_W(l);
            for(int i = 0; i < fan_in * WIDTH; ++i) P[o + i] = (float)ud(rng);
        }
    }
    MCHECK(hipMemcpy(m->P, P.data(), np * 4, hipMemcpyHostToDevice));
    MCHECK(hipMemcpy(m->Bf, Bf.data(), Bf.size() * 4, hipMemcpyHostToDevice));
    MCHECK(hipMemset(m->Mo, 0, np * 4));
    MCHECK(hipMemset(m->Vo, 0, np * 4));
    refresh_bf(m);
    MCHECK(hipGetLastError());
    MCHECK(hipStreamSynchronize(m->stream));
    *out = m;
    return 0;
}

// A coordinate network (one output, Fourier front).
extern "C" int bhc_mlp_create(int device, int members, int max_batch, unsigned long long seed, float sigma,
                              bhc_mlp **out)
{
    return bhc_mlp_create_ex(device, members, max_batch, 1, 0, seed, sigma, out);
}

extern "C" int bhc_mlp_get_params(bhc_mlp *m, float *params, float *fourier)
{
    MCHECK(hipSetDevice(m->device));
    MCHECK(hipStreamSynchronize(m->stream));
    if(params) MCHECK(hipMemcpy(params, m->P, (size_t)m->members * m->np * 4, hipMemcpyDeviceToHost));
    if(fourier) MCHECK(hipMemcpy(fourier, m->Bf, N_FREQ * D_IN * 4, hipMemcpyDeviceToHost));
    return 0;
}

// Replace the Fourier projection matrix B [32][16] (features sin / cos of
// 2 pi B x), e.g. with per-input frequency scales.
extern "C" int bhc_mlp_set_fourier(bhc_mlp *m, const float *B)
{
    MCHECK(hipSetDevice(m->device));
    MCHECK(hipMemcpy(m->Bf, B, N_FREQ * D_IN * 4, hipMemcpyHostToDevice));
    return 0;
}

extern "C" int bhc_mlp_set_params(bhc_mlp *m, const float *params)
{
    MCHECK(hipSetDevice(m->device));
    size_t np = (size_t)m->members * m->np;
    MCHECK(hipMemcpy(m->P, params, np * 4, hipMemcpyHostToDevice));
    refresh_bf(m);
    MCHECK(hipGetLastError());
    MCHECK(hipStreamSynchronize(m->stream));
    return 0;
}

// Predictions of every member for n points x[n][16] (host); out[members][n][n_out].
extern "C" int bhc_mlp_predict(bhc_mlp *m, const float *x, long long n, float *out)
{
    MCHECK(hipSetDevice(m->device));
    const int K = m->n_out;
    for(long long b0 = 0; b0 < n; b0 += m->max_batch) {
        int nb = (int)std::min<long long>(m->max_batch, n - b0);
        MCHECK(hipMemcpyAsync(m->x, x + b0 * D_IN, (size_t)nb * D_IN * 4, hipMemcpyHostToDevice, m->stream));
        forward(m, m->x, nb);
        MCHECK(hipGetLastError());
        // one copy where the members' results are adjacent in the caller's array too
        const int parts = nb == n ? 1 : m->members;
        const size_t len = (size_t)(nb == n ? m->members : 1) * nb * K;
        for(int e = 0; e < parts; ++e)
            MCHECK(hipMemcpyAsync(out + ((size_t)e * n + b0) * K, m->out + e * len, len * 4, hipMemcpyDeviceToHost,
                                  m->stream));
        MCHECK(hipStreamSynchronize(m->stream));
    }
    return 0;
}

// Gradients (FP32, [members][params]) and per-member loss for one batch
// (n <= max_batch points, x [n][16], y [n][n_out], host arrays), without
// updating the weights.
extern "C" int bhc_mlp_gradients(bhc_mlp *m, const float *x, const float *y, int n, float *grads, float *loss)
{
    if(n < 1 || n > m->max_batch || n % 32) return mfail("bhc_mlp_gradients: n must be a multiple of 32 <= max_batch");
    MCHECK(hipSetDevice(m->device));
    MCHECK(hipMemcpyAsync(m->x, x, (size_t)n * D_IN * 4, hipMemcpyHostToDevice, m->stream));
    MCHECK(hipMemcpyAsync(m->y, y, (size_t)n * m->n_out * 4, hipMemcpyHostToDevice, m->stream));
    zero_grads(m);
    m->last_loss = 0;
    forward_backward(m, m->x, m->y, nullptr, n, m->loss);
    MCHECK(hipGetLastError());
    if(grads)
        MCHECK(hipMemcpyAsync(grads, m->G, (size_t)m->members * m->np * 4, hipMemcpyDeviceToHost, m->stream));
    if(loss) MCHECK(hipMemcpyAsync(loss, m->loss, (size_t)m->members * 4, hipMemcpyDeviceToHost, m->stream));
    MCHECK(hipStreamSynchronize(m->stream));
    return 0;
}

// Resident training set: X[n][16] normalised inputs, Y[n][n_out] normalised targets.
extern "C" int bhc_mlp_set_dataset(bhc_mlp *m, const float *X, const float *Y, long long n)
{
    MCHECK(hipSetDevice(m->device));
    if(m->X) (void)hipFree(m->X);
    if(m->Y) (void)hipFree(m->Y);
    m->X = m->Y = nullptr;
    MCHECK(bhc_device_malloc((void **)&m->X, (size_t)n * D_IN * 4));
    MCHECK(bhc_device_malloc((void **)&m->Y, (size_t)n * m->n_out * 4));
    MCHECK(hipMemcpy(m->X, X, (size_t)n * D_IN * 4, hipMemcpyHostToDevice));
    MCHECK(hipMemcpy(m->Y, Y, (size_t)n * m->n_out * 4, hipMemcpyHostToDevice));
    m->nset = n;
    return 0;
}

// `steps` Adam steps on batches of `batch` points drawn (with replacement,
// from `seed`) from the resident training set. loss_out[members]: mean loss
// of the last step. The steps run back to back on the GPU; the kernel time
// is kept for bhc_mlp_last_ms.
extern "C" int bhc_mlp_train(bhc_mlp *m, int steps, int batch, float lr, unsigned long long seed, float *loss_out)
{
    if(!m->X || batch < 32 || batch > m->max_batch || batch % 32) return mfail("bhc_mlp_train: bad batch or no dataset");
    MCHECK(hipSetDevice(m->device));
    std::mt19937_64 rng(seed);
    std::uniform_int_distribution<long long> ud(0, m->nset - 1);
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    MCHECK(hipEventRecord(m->e0, m->stream));
    if(steps > 0) zero_grads(m);
    // batches are drawn a chunk of steps at a time, while the GPU works on the
    // chunk before; the copy follows that chunk's steps on the stream
    std::vector<int32_t> idx((size_t)steps * batch);
    for(int s0 = 0; s0 < steps; s0 += IDX_CHUNK) {
        const int ns = std::min(IDX_CHUNK, steps - s0);
        int32_t *chunk = idx.data() + (size_t)s0 * batch;
        for(size_t i = 0; i < (size_t)ns * batch; ++i) chunk[i] = (int32_t)ud(rng);
        MCHECK(hipMemcpyAsync(m->idx, chunk, (size_t)ns * batch * 4, hipMemcpyHostToDevice, m->stream));
        for(int s = 0; s < ns; ++s) {
            float *loss = m->loss + 16 * ((s0 + s) & 1), *next = m->loss + 16 * ((s0 + s + 1) & 1);
            forward_backward(m, m->X, m->Y, m->idx + (size_t)s * batch, batch, loss);
            m->last_loss = (s0 + s) & 1;
            ++m->step;
            float c1 = 1.0f - std::pow(b1, (float)m->step), c2 = 1.0f - std::pow(b2, (float)m->step);
            hipLaunchKernelGGL(k_adam<true>, dim3(n_tiles(m->n_out) + (n_loose(m->n_out) + 255) / 256, m->members),
                               dim3(256), 0, m->stream, m->P, m->Mo, m->Vo, m->G, m->Wf, m->Wb, m->np, m->npf, m->n_out,
                               lr, b1, b2, eps, c1, c2, next);
        }
    }
    MCHECK(hipEventRecord(m->e1, m->stream));
    MCHECK(hipGetLastError());
    if(loss_out)
        MCHECK(hipMemcpyAsync(loss_out, m->loss + 16 * m->last_loss, (size_t)m->members * 4, hipMemcpyDeviceToHost, m->stream));
    MCHECK(hipStreamSynchronize(m->stream));
    float ms = 0.f;
    MCHECK(hipEventElapsedTime(&ms, m->e0, m->e1));
    m->last_ms = ms;
    return 0;
}

extern "C" double bhc_mlp_last_ms(bhc_mlp *m) { return m ? m->last_ms : 0.0; }

// Matrix-core FLOPs of one training step on `batch` points (forward +
// backward products of the hidden layers and, with several outputs, of the
// output layer; all members).
extern "C" double bhc_mlp_step_flops(bhc_mlp *m, int batch)
{
    double f = 0.0;
    for(int l = 0; l < N_HID; ++l) {
        double k = l == 0 ? D_FF : WIDTH;
        f += 2.0 * batch * k * WIDTH * (l == 0 ? 2.0 : 3.0); // forward, dW, (dH for l > 0)
    }
    if(m->n_out > 1) f += 2.0 * batch * WIDTH * m->n_out * 3.0;
    return f * m->members;
}
