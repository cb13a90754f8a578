// Learned directional proposal: network kernels on the matrix cores and the
// dl_hip_guide_* entry points.
//
// Every GEMM of the 96-64-64-64-64-48 network runs as 32x32x16 bfloat16 MFMA
// tiles with float32 accumulation (v_mfma_f32_32x32x16_bf16).  Operand lane
// layout (checked on the device): lane l holds A[l%32][(l/32)*8 + 0..7] and
// B[(l/32)*8 + 0..7][l%32]; accumulator register r of lane l is
// D[8*(r/4) + 4*(l/32) + (r%4)][l%32].
//
//   forward     a wave takes 64 rows (two 32-row blocks); activations live
//               in the wave's LDS rows (bfloat16, in place layer by layer);
//               weights are read from global memory (43 KB, L2-resident) as
//               A operands, 1 KB in a row per tile
//   training    one kernel per step for forward, loss and backward (16x16x32
//               and 32x32x16 tiles): a block keeps its rows' activations in LDS
//               and its share of dW in registers; per-block partial gradients are then summed in a
//               fixed order, with Adam in the same kernel (float32 master
//               weights; the bfloat16 copies of W and W^T, laid out in the
//               order in which the operands are read, are refreshed there)
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../render_sizes.h"
#include "backend.h"
#include "guide.h"

namespace dl {

namespace {

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));  // a caller's rows

// Network evaluation on float32 inputs x (n x 96).
__global__ __launch_bounds__(kGWaves * 64) void k_mlp_forward(Net net, const float* __restrict__ x, uint32_t n,
                                                             float* __restrict__ out) {
    __shared__ __align__(16) uint16_t s_act[kGWaves][kGRowsPerWave * kGRowStride];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint16_t* s = s_act[wave];
    for (uint32_t tile = blockIdx.x * kGWaves + wave; (size_t)tile * kGRowsPerWave < n; tile += gridDim.x * kGWaves) {
        const uint32_t row0 = tile * kGRowsPerWave;
        const uint32_t row = row0 + lane;
        float f[8];
        for (int q = 0; q < kGIn / 8; q++) {
            for (int j = 0; j < 8; j++) f[j] = row < n ? x[(size_t)row * kGIn + q * 8 + j] : 0.0f;
            *reinterpret_cast<bf16x8*>(s + lane * kGRowStride + q * 8) = pack8(f);
        }
        forward_rows(net, s, [&](int r, int c, float4 v) {
            if (row0 + r < n)
                *reinterpret_cast<f32x4_any*>(out + (size_t)(row0 + r) * kGOut + c) = f32x4_any{v.x, v.y, v.z, v.w};
        });
    }
}

// Raw outputs -> mixture parameters (n x 40).
__global__ void k_mlp_decode(const float* __restrict__ out, uint32_t n, float* __restrict__ mix) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float o[kGOut], m[kGMix];
        for (int j = 0; j < kGOut; j++) o[j] = out[(size_t)i * kGOut + j];
        guide_decode(o, m);
        for (int j = 0; j < kGMix; j++) mix[(size_t)i * kGMix + j] = m[j];
    }
}

// Sum of a 256-thread block's values, in every thread of the first wave.
__device__ __forceinline__ float block_sum(float v) {
    __shared__ float s_part[4];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = v;
    __syncthreads();
    return (s_part[0] + s_part[1]) + (s_part[2] + s_part[3]);
}

// Partial sums of the training weights, one per block (kSumBlocks blocks),
// which every training block adds in the same order.
__global__ __launch_bounds__(256) void k_sum(const float* __restrict__ c, uint32_t n, float* __restrict__ part) {
    float acc = 0.0f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) acc += c[i];
    acc = block_sum(acc);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// ---- one training step's forward, loss and backward -----------------------
// loss = sum(-c log q(d)) / sum(c) and its gradient.  Each of a block's four
// waves takes 16 rows of a 64-row tile through the network and back:
//
//   forward   D[out][row] = W act^T + b per layer (16x16x32): a lane's
//             accumulators are one row's outputs in runs of four, so the next
//             layer's operand rows are written 8 bytes at a time; every
//             layer's inputs are also kept transposed ([column][row]) for dW
//   loss      four lanes per row, two lobes each; dLoss/dout in registers
//   backward  per layer, from the output: dW[out][in] += g^T act over the
//             tile's 64 rows (22 tiles of 32x32 shared out over the waves,
//             accumulated in registers over the block's whole run), and
//             D[in][row] = W^T g^T with the ReLU mask the forward left in
//             registers, in the same layout again
//
// The bias gradients are summed from the unrounded float32 gradients; what the
// matrix products read is bfloat16, as in the forward.  Two blocks per CU (73
// KB of LDS and up to 256 registers each).  What bounds it is latency: each
// wave's chain of LDS and matrix steps, and the weights, read per tile from L1/L2: 144 us for 2^18 rows,
// 0.23 PFLOP/s (249 us with the weights' pointers laundered into flat loads,
// which also wait for the LDS, and a wait at each change of LDS type).  A step
// of 2^18 rows took 814 us as fifteen launches (forward, loss, and dW, its
// reduction and dAct per layer, 700 bytes of activations and gradients per row
// through memory) and takes 208 us as three.
constexpr int kTrainWaves = 4, kTrainRows = 16 * kTrainWaves;
static_assert(kTrainRows == (int)dl_sizes::kGuideTrainRows, "rows of a training tile");
constexpr int kTrainStride = kTrainRows + 8;         // bf16 per transposed column
constexpr int kTrainCols = kGIn + 4 * kGHid;         // the inputs of the five layers
constexpr int kTrainOutStride = kGOut + 1;           // float32 outputs of a row
constexpr int kSumBlocks = (int)dl_sizes::kGuideSumBlocks;
static_assert(kSumBlocks == 64, "one partial sum per lane");
static_assert(kTrainOutStride * 4 <= kGRowStride * 2, "outputs overlay the operand rows");
constexpr int train_col(int l) { return l == 0 ? 0 : kGIn + (l - 1) * kGHid; }

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
    // lane l holds A[l%16][(l/16)*8 + 0..7] and B[(l/16)*8 + 0..7][l%16];
    // register r of the result is D[4*(l/16) + r][l%16]
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
}
// Sums over the 16 rows of a wave (lanes of equal quad) of each of a lane's 16
// values: lane rl returns the sum of value rl (v[rl / 4][rl % 4]).  Four
// exchange steps, each halving the values: lanes l and l ^ 8, l ^ 7, l ^ 2,
// l ^ 1.  (Kept per lane until the end, the sums of the hidden layers' biases
// took 64 registers, and the accumulators spilled.)
template <int CTRL, int CNT>
__device__ __forceinline__ void row_sum_step(float (&a)[16], bool up) {
#pragma unroll
    for (int i = 0; i < CNT; i++) {
        const float keep = up ? a[i + CNT] : a[i], send = up ? a[i] : a[i + CNT];
        a[i] = keep + __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(send), CTRL, 0xf, 0xf, true));
    }
}
__device__ __forceinline__ float row_sums(const float (&v)[4][4], int rl) {
    float a[16];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) a[4 * t + r] = v[t][r];
    row_sum_step<0x128, 8>(a, (rl & 8) != 0);  // row_ror:8
    row_sum_step<0x141, 4>(a, (rl & 4) != 0);  // row_half_mirror
    row_sum_step<0x4e, 2>(a, (rl & 2) != 0);   // quad_perm [2, 3, 0, 1]
    row_sum_step<0xb1, 1>(a, (rl & 1) != 0);   // quad_perm [1, 0, 3, 2]
    return a[0];
}

// A lane's 16 values of a row (four tiles of four, accumulator layout) as
// bfloat16: into the row's operand row and the transposed columns.
__device__ __forceinline__ void put_row(const float (&v)[4][4], int quad, uint16_t* __restrict__ row,
                                        uint16_t* __restrict__ col) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int c = 16 * t + 4 * quad;
        const uint32_t a = pack2(v[t][0], v[t][1]), b = pack2(v[t][2], v[t][3]);
        *reinterpret_cast<uint2*>(row + c) = make_uint2(a, b);
        uint16_t* k = col + c * kTrainStride;
        k[0] = (uint16_t)a;
        k[kTrainStride] = (uint16_t)(a >> 16);
        k[2 * kTrainStride] = (uint16_t)b;
        k[3 * kTrainStride] = (uint16_t)(b >> 16);
    }
}

__global__ __launch_bounds__(kTrainWaves * 64, 2) void k_train(Net net, const float* __restrict__ x,
                                                             const float* __restrict__ dirs,
                                                             const float* __restrict__ cw, uint32_t n,
                                                             const float* __restrict__ sums, float* __restrict__ part,
                                                             float* __restrict__ loss) {
    __shared__ __align__(16) uint16_t s_col[kTrainCols * kTrainStride];      // layer inputs, transposed
    __shared__ __align__(16) uint16_t s_g[kGHid * kTrainStride];             // a layer's gradients, transposed
    __shared__ __align__(16) uint16_t s_row[kTrainWaves][16 * kGRowStride];  // each wave's operand rows
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int rl = lane & 15, quad = lane >> 4;   // row and column group of the 16-row products
    const int rl32 = lane & 31, half = lane >> 5;  // of the 32x32 tiles of dW
    uint16_t* const myrow = s_row[wave] + rl * kGRowStride;
    float* const outs = reinterpret_cast<float*>(s_row[wave]) + rl * kTrainOutStride;
    const int trow = wave * 16 + rl;  // the lane's row of the tile
    float invc;
    {
        float t = sums[lane];
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off);
        invc = 1.0f / fmaxf(t, 1e-30f);
    }
    f32x16 dw[6];  // 0, 1: layer 0 (the second in waves 0 and 1 only); 1 + l: layer l
#pragma unroll
    for (int k = 0; k < 6; k++) dw[k] = f32x16{0};
    // bias sums: of the hidden layers over the wave's rows (row_sums), of the
    // output layer over the lane's
    float db[4] = {0.f, 0.f, 0.f, 0.f}, db4[10], lacc = 0.0f;
#pragma unroll
    for (int j = 0; j < 10; j++) db4[j] = 0.0f;

    const uint32_t tiles = (n + kTrainRows - 1) / kTrainRows;
    const uint32_t share = (tiles + gridDim.x - 1) / gridDim.x;  // consecutive tiles of a block
    const uint32_t end = blockIdx.x < tiles / share ? (blockIdx.x + 1) * share : tiles;
    for (uint32_t tile = blockIdx.x * share; tile < end; tile++) {
        const uint32_t row = tile * kTrainRows + trow;
        const bool valid = row < n;
        // (the weights are read again for each tile: kept in registers over the
        // loop, they would push the accumulators to scratch memory)
        uint32_t again = 0;
        asm volatile("" : "+s"(again));
        const uint16_t *w_all = net.w16 + again, *wt_all = net.wt16 + again;
        const float* b_all = net.bias + again;
        // ---- inputs
        f32x4 xin[6];
        vec3 d = v3(0.f, 0.f, 1.f);
        float ci = 0.0f;
        if (valid) {
            const f32x4_any* src = reinterpret_cast<const f32x4_any*>(x + (size_t)row * kGIn) + quad;
#pragma unroll
            for (int q = 0; q < 6; q++) xin[q] = src[4 * q];
            d = v3(dirs[3 * (size_t)row], dirs[3 * (size_t)row + 1], dirs[3 * (size_t)row + 2]);
            ci = cw[row];
        } else {
#pragma unroll
            for (int q = 0; q < 6; q++) xin[q] = f32x4{0};
        }
        __syncthreads();  // the previous tile's columns have been read
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const int c = 16 * q + 4 * quad;
            const uint32_t a = pack2(xin[q].x, xin[q].y), b = pack2(xin[q].z, xin[q].w);
            *reinterpret_cast<uint2*>(myrow + c) = make_uint2(a, b);
            uint16_t* k = s_col + c * kTrainStride + trow;
            k[0] = (uint16_t)a;
            k[kTrainStride] = (uint16_t)(a >> 16);
            k[2 * kTrainStride] = (uint16_t)b;
            k[3 * kTrainStride] = (uint16_t)(b >> 16);
        }
        lds_order();
        // ---- forward
        uint32_t mask[4];  // ReLU of layers 0..3: bit 4 t + r
        float v[4][4];
#pragma unroll
        for (int l = 0; l < 5; l++) {
            constexpr int kK[5] = {kGIn, kGHid, kGHid, kGHid, kGHid};
            const int T = l < 4 ? 4 : kGOut / 16;
            const uint16_t* W = w_all + l * kGWSlot + lane * 8;
            const float4* bias = reinterpret_cast<const float4*>(b_all + l * 64) + quad;
            f32x4 acc[4];
#pragma unroll
            for (int t = 0; t < 4; t++) acc[t] = f32x4{0};
#pragma unroll
            for (int kt = 0; kt < kK[l] / 32; kt++) {
                const bf16x8 b = *reinterpret_cast<const bf16x8*>(myrow + kt * 32 + quad * 8);
#pragma unroll
                for (int t = 0; t < T; t++)
                    acc[t] = mfma16(*reinterpret_cast<const bf16x8*>(W + (t * (kK[l] / 32) + kt) * 512), b, acc[t]);
            }
            lds_order();
            uint32_t m = 0;
#pragma unroll
            for (int t = 0; t < T; t++) {
                const float4 b4 = bias[4 * t];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float a = acc[t][r] + (r == 0 ? b4.x : r == 1 ? b4.y : r == 2 ? b4.z : b4.w);
                    v[t][r] = l < 4 ? fmaxf(a, 0.0f) : a;
                    if (l < 4) m |= a > 0.0f ? 1u << (4 * t + r) : 0u;
                }
            }
            if (l < 4) {
                mask[l] = m;
                put_row(v, quad, myrow, s_col + train_col(l + 1) * kTrainStride + trow);
                lds_order();
            }
        }
        // ---- loss
#pragma unroll
        for (int t = 0; t < kGOut / 16; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) outs[16 * t + 4 * quad + r] = v[t][r];
        lds_order();
        float o[10], gl[10];
#pragma unroll
        for (int j = 0; j < 10; j++) o[j] = outs[10 * quad + j];
        lds_order();
        {
            auto over_quads = [](float a) {
                a += __shfl_xor(a, 16);
                return a + __shfl_xor(a, 32);
            };
            float mx = fmaxf(o[0], o[5]);
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            float e[2];
#pragma unroll
            for (int j = 0; j < 2; j++) e[j] = expf(o[5 * j] - mx);
            const float sum = over_quads(e[0] + e[1]);
            float w[2], kap[2], sg[2], nm[2], dt[2], f[2];
            vec3 mu[2];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                w[j] = e[j] / sum;
                sg[j] = 1.0f / (1.0f + expf(-o[5 * j + 1]));
                kap[j] = expf(kGKappaLo + (kGKappaHi - kGKappaLo) * sg[j]);
                const float a = o[5 * j + 2], b = o[5 * j + 3], c = o[5 * j + 4];
                nm[j] = fmaxf(sqrtf(a * a + b * b + c * c), 1e-6f);
                mu[j] = v3(a / nm[j], b / nm[j], c / nm[j]);
                dt[j] = dot(mu[j], d);
                f[j] = vmf_pdf(kap[j], mu[j], d);
            }
            const float q = over_quads(w[0] * f[0] + w[1] * f[1]);
            const float qs = fmaxf(q, 1e-30f);
            if (quad == 0) lacc += -ci * logf(qs) * invc;
            const float gq = -ci / qs * invc;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float wf = w[j] * f[j], k = kap[j];
                gl[5 * j] = gq * (wf - w[j] * q);
                const float em = -expm1f(-2.0f * k);
                const float dlogf = 1.0f / k - 2.0f * expf(-2.0f * k) / em + (dt[j] - 1.0f);
                gl[5 * j + 1] = gq * wf * dlogf * k * (kGKappaHi - kGKappaLo) * sg[j] * (1.0f - sg[j]);
                const float s = gq * wf * k / nm[j];
                gl[5 * j + 2] = s * (d.x - dt[j] * mu[j].x);
                gl[5 * j + 3] = s * (d.y - dt[j] * mu[j].y);
                gl[5 * j + 4] = s * (d.z - dt[j] * mu[j].z);
            }
        }
#pragma unroll
        for (int j = 0; j < 10; j += 2) {
            db4[j] += gl[j];
            db4[j + 1] += gl[j + 1];
            const uint32_t a = pack2(gl[j], gl[j + 1]);
            const int c = 10 * quad + j;
            *reinterpret_cast<uint32_t*>(myrow + c) = a;
            s_g[c * kTrainStride + trow] = (uint16_t)a;
            s_g[(c + 1) * kTrainStride + trow] = (uint16_t)(a >> 16);
        }
        // columns 40..47 carry no output (gradient zero), 48..63 pad the product
        // (their dW is discarded)
#pragma unroll
        for (int j = 0; j < 6; j += 2) *reinterpret_cast<uint32_t*>(myrow + kGMix + 6 * quad + j) = 0u;
#pragma unroll
        for (int j = 0; j < 2; j++) s_g[(kGMix + 2 * quad + j) * kTrainStride + trow] = 0;
        // ---- backward
#pragma unroll
        for (int l = 4; l >= 0; l--) {
            __syncthreads();  // every wave's rows of s_g are there
            auto dw_tile = [&](int ot, int it, f32x16& acc) {
                const uint16_t* A = s_g + (ot * 32 + rl32) * kTrainStride + half * 8;
                const uint16_t* B = s_col + (train_col(l) + it * 32 + rl32) * kTrainStride + half * 8;
#pragma unroll
                for (int kt = 0; kt < kTrainRows / 16; kt++)
                    acc = mfma(*reinterpret_cast<const bf16x8*>(A + kt * 16),
                               *reinterpret_cast<const bf16x8*>(B + kt * 16), acc);
            };
            if (l > 0) {
                dw_tile(wave >> 1, wave & 1, dw[1 + l]);
                const uint16_t* WT = wt_all + l * kGWSlot + lane * 8;
                f32x4 acc[4];
#pragma unroll
                for (int t = 0; t < 4; t++) acc[t] = f32x4{0};
#pragma unroll
                for (int kt = 0; kt < 2; kt++) {
                    const bf16x8 b = *reinterpret_cast<const bf16x8*>(myrow + kt * 32 + quad * 8);
#pragma unroll
                    for (int t = 0; t < 4; t++)
                        acc[t] = mfma16(*reinterpret_cast<const bf16x8*>(WT + (2 * t + kt) * 512), b, acc[t]);
                }
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) v[t][r] = (mask[l - 1] >> (4 * t + r)) & 1u ? acc[t][r] : 0.0f;
                db[l - 1] += row_sums(v, rl);
                __syncthreads();  // dW has read s_g
                put_row(v, quad, myrow, s_g + trow);
            } else {
                dw_tile(wave / 3, wave % 3, dw[0]);
                if (wave < 2) dw_tile(1, wave + 1, dw[1]);
            }
        }
    }
    // ---- the block's partial gradient
    float* const dst = part + (size_t)blockIdx.x * kGParams;
    auto put_dw = [&](int l, int ot, int it, const f32x16& acc) {
        const int K = glayer_in(l);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int o = ot * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (o < glayer_out(l)) dst[glayer_w(l) + o * K + it * 32 + rl32] = acc[r];
        }
    };
    put_dw(0, wave / 3, wave % 3, dw[0]);
    if (wave < 2) put_dw(0, 1, wave + 1, dw[1]);
#pragma unroll
    for (int l = 1; l < 5; l++) put_dw(l, wave >> 1, wave & 1, dw[1 + l]);
    // bias sums: over the wave's rows, then over the waves
    __syncthreads();
    float* const s_b = reinterpret_cast<float*>(s_col);  // [wave][5][64], then the losses
    auto over_rows = [](float a) {
        for (int off = 8; off > 0; off >>= 1) a += __shfl_xor(a, off);
        return a;
    };
#pragma unroll
    for (int l = 0; l < 4; l++) s_b[(wave * 5 + l) * 64 + 16 * (rl >> 2) + 4 * quad + (rl & 3)] = db[l];
#pragma unroll
    for (int j = 0; j < 10; j++) {
        const float a = over_rows(db4[j]);
        if (rl == 0) s_b[(wave * 5 + 4) * 64 + 10 * quad + j] = a;
    }
    if (quad == 0 && rl < kGOut - kGMix) s_b[(wave * 5 + 4) * 64 + kGMix + rl] = 0.0f;
    lacc = over_rows(lacc);
    if (lane == 0) s_b[kTrainWaves * 5 * 64 + wave] = lacc;
    __syncthreads();
    for (int k = threadIdx.x; k < 5 * 64; k += kTrainWaves * 64) {
        const int l = k >> 6, o = k & 63;
        if (o < glayer_out(l))
            dst[glayer_b(l) + o] = (s_b[k] + s_b[5 * 64 + k]) + (s_b[10 * 64 + k] + s_b[15 * 64 + k]);
    }
    if (threadIdx.x == 0) {
        const float* w = s_b + kTrainWaves * 5 * 64;
        loss[blockIdx.x] = (w[0] + w[1]) + (w[2] + w[3]);
    }
}

// A parameter's float32 value to the network's bfloat16 copies and biases.
__device__ __forceinline__ void refresh_param(int idx, float th, uint16_t* __restrict__ w, uint16_t* __restrict__ w16,
                                              uint16_t* __restrict__ wt16, float* __restrict__ bias) {
    int l = 4;
    while (l > 0 && idx < glayer_w(l)) l--;
    const int K = glayer_in(l), off = idx - glayer_w(l);
    if (off < glayer_out(l) * K) {
        const int o = off / K, i = off % K;
        w[l * kGWSlot + operand_index(o, i, K)] = f2bf(th);
        w16[l * kGWSlot + operand16_index(o, i, K)] = f2bf(th);
        wt16[l * kGWSlot + operand16_index(i, o, 64)] = f2bf(th);
    } else {
        bias[l * 64 + (off - glayer_out(l) * K)] = th;
    }
}

__global__ void k_refresh(const float* __restrict__ theta, uint16_t* __restrict__ w, uint16_t* __restrict__ w16,
                          uint16_t* __restrict__ wt16, float* __restrict__ bias) {
    for (int idx = blockIdx.x * blockDim.x + threadIdx.x; idx < kGParams; idx += gridDim.x * blockDim.x)
        refresh_param(idx, theta[idx], w, w16, wt16, bias);
}

// grad[e] += sum over blocks of part[block][e], and with `apply` the Adam
// update of parameter e from it; the step's loss from the blocks' losses.
// Block: 64 parameters, read 16 bytes a lane, x 16 groups of partials (group q
// sums blocks q, q + 16, ...); everything is added in a fixed order.  Bound by
// the reads of the partials: 512 of 21,808 parameters (45 MB): 12.6 us.
// With four groups of 4-byte reads a thread had 128 dependent additions and few
// reads in flight: 39 us.
constexpr int kReduceGroups = 16;
struct AdamArgs {
    float *theta, *m, *v, *grad;
    float lr, c1, c2;
    int apply;
    uint16_t *w, *w16, *wt16;
    float* bias;
};
__global__ __launch_bounds__(256) void k_train_reduce(const float* __restrict__ part, uint32_t blocks, AdamArgs a,
                                                      const float* __restrict__ block_loss, float* __restrict__ loss) {
    static_assert(kGParams % 4 == 0, "the partials are read in float4");
    __shared__ __align__(16) float s_sum[kReduceGroups][64];
    const uint32_t q = threadIdx.x >> 4, e4 = blockIdx.x * 64 + 4 * (threadIdx.x & 15);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (e4 < (uint32_t)kGParams) {
        const float* src = part + e4;
#pragma unroll 8
        for (uint32_t b = q; b < blocks; b += kReduceGroups) {
            const float4 t = *reinterpret_cast<const float4*>(src + (size_t)b * kGParams);
            v.x += t.x;
            v.y += t.y;
            v.z += t.z;
            v.w += t.w;
        }
    }
    *reinterpret_cast<float4*>(&s_sum[q][4 * (threadIdx.x & 15)]) = v;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const uint32_t e = blockIdx.x * 64 + threadIdx.x;
    if (blockIdx.x == 0) {
        float t = 0.0f;
        for (uint32_t b = threadIdx.x; b < blocks; b += 64) t += block_loss[b];
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off);
        if (threadIdx.x == 0) *loss = t;
    }
    if (e >= (uint32_t)kGParams) return;
    float sum[kReduceGroups];
#pragma unroll
    for (int k = 0; k < kReduceGroups; k++) sum[k] = s_sum[k][threadIdx.x];
#pragma unroll
    for (int n = 1; n < kReduceGroups; n *= 2)
#pragma unroll
        for (int k = 0; k < kReduceGroups; k += 2 * n) sum[k] += sum[k + n];
    const float gr = a.grad[e] + sum[0];
    if (!a.apply) {
        a.grad[e] = gr;
        return;
    }
    const float mm = 0.9f * a.m[e] + 0.1f * gr;
    const float vv = 0.999f * a.v[e] + 0.001f * gr * gr;
    a.m[e] = mm;
    a.v[e] = vv;
    const float th = a.theta[e] - a.lr * (mm / a.c1) / (sqrtf(vv / a.c2) + 1e-8f);
    a.theta[e] = th;
    a.grad[e] = 0.0f;
    refresh_param((int)e, th, a.w, a.w16, a.wt16, a.bias);
}

// Training weight of one render record: c = L_i(d) / p(d), the incident
// radiance estimated from the path's final radiance as (L_final - L_before)
// / T (T: throughput after the vertex, per channel, averaged over the
// channels with T > 0), divided by the density d was sampled from.  Zero
// for an empty slot, a non-finite estimate or a non-finite direction.
__device__ __forceinline__ float record_weight(const float* __restrict__ q, const float4* __restrict__ rad) {
    if (q[kRecValid] == 0.0f) return 0.0f;
    const uint32_t p = __float_as_uint(q[kRecPath]);
    const float4 rf = rad[p];
    const float fin[3] = {rf.x, rf.y, rf.z};
    float sum = 0.0f;
    int cnt = 0;
    for (int k = 0; k < 3; k++) {
        const float t = q[kRecThr + k];
        if (t > 0.0f) {
            sum += (fin[k] - q[kRecRad + k]) / t;
            cnt++;
        }
    }
    const float pdf = q[kRecPdf];
    float w = (cnt > 0 && pdf > 0.0f) ? (sum / (float)cnt) / pdf : 0.0f;
    if (!(w >= 0.0f) || !isfinite(w)) w = 0.0f;
    if (!isfinite(q[kRecDir]) || !isfinite(q[kRecDir + 1]) || !isfinite(q[kRecDir + 2])) w = 0.0f;
    return w;
}

// Batch row r from record q with weight w (features zeroed when w == 0).
__device__ __forceinline__ void write_batch_row(const float* __restrict__ q, float w, uint32_t r, float* __restrict__ x,
                                                float* __restrict__ d, float* __restrict__ c) {
    const vec3 pn = v3(q[kRecPos], q[kRecPos + 1], q[kRecPos + 2]);
    const vec3 wo = v3(q[kRecWo], q[kRecWo + 1], q[kRecWo + 2]);
    const vec3 nn = v3(q[kRecN], q[kRecN + 1], q[kRecN + 2]);
    for (int ch = 0; ch < kGIn / 8; ch++) {
        float f[8];
        if (w > 0.0f)
            guide_feature_chunk(pn, wo, nn, q[kRecRough], ch, f);
        else
            for (int j = 0; j < 8; j++) f[j] = 0.0f;
        for (int j = 0; j < 8; j++) x[(size_t)r * kGIn + ch * 8 + j] = f[j];
    }
    const bool ok = w > 0.0f;
    d[3 * r] = ok ? q[kRecDir] : 0.0f;
    d[3 * r + 1] = ok ? q[kRecDir + 1] : 0.0f;
    d[3 * r + 2] = ok ? q[kRecDir + 2] : 1.0f;
    c[r] = w;
}

// ---- resampling of records in proportion to their weights ----------------
// The batch gradient sum_r c_r grad(-log q(d_r)) / sum_r c_r equals in
// expectation the mean of grad(-log q(d)) over records drawn with
// probability c_r / sum c; drawing them (systematic resampling over the
// weights' prefix sums) gives every batch row weight 1, so one batch spends
// its rows on the records that carry radiance.
constexpr int kScanThreads = 256, kScanItems = 4, kScanTile = kScanThreads * kScanItems;

// Record weights, each capped at `share` of *total when total is given (a
// rare path of enormous weight would otherwise fill whole batches with
// copies of itself).
__global__ void k_record_weights(const float* __restrict__ rec, uint32_t R, const float4* __restrict__ rad,
                                 const float* __restrict__ total, float share, float* __restrict__ w) {
    const float cap = total ? share * *total : INFINITY;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < R; r += gridDim.x * blockDim.x)
        w[r] = fminf(record_weight(rec + (size_t)r * kGRecFloats, rad), cap);
}

// In-place inclusive prefix sums of each kScanTile-element tile of w; the
// tile totals to tile_sum.  Fixed summation order (deterministic).
__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(float* __restrict__ w, uint32_t R,
                                                             float* __restrict__ tile_sum) {
    __shared__ float s_wave[kScanThreads / 64];
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float v[kScanItems];
    float run = 0.0f;
    for (int k = 0; k < kScanItems; k++) {
        run += base + k < R ? w[base + k] : 0.0f;
        v[k] = run;
    }
    float x = run;
    for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    float woff = 0.0f;
    for (int j = 0; j < wave; j++) woff += s_wave[j];
    const float excl = woff + (x - run);
    for (int k = 0; k < kScanItems; k++)
        if (base + k < R) w[base + k] = excl + v[k];
    if (threadIdx.x == kScanThreads - 1) tile_sum[blockIdx.x] = woff + x;
}

// Exclusive prefix of the tile totals: tile_off[b] = sum of tiles < b,
// tile_off[nt] = the grand total.  One block; each thread sums a run of
// tiles serially, then one thread prefixes the runs.
__global__ __launch_bounds__(kScanThreads) void k_scan_top(const float* __restrict__ tile_sum, uint32_t nt,
                                                           float* __restrict__ tile_off) {
    __shared__ float s_run[kScanThreads];
    const uint32_t per = (nt + kScanThreads - 1) / kScanThreads;
    const uint32_t b0 = threadIdx.x * per;
    float acc = 0.0f;
    for (uint32_t b = b0; b < b0 + per && b < nt; b++) acc += tile_sum[b];
    s_run[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (int j = 0; j < kScanThreads; j++) {
            const float a = s_run[j];
            s_run[j] = t;
            t += a;
        }
        tile_off[nt] = t;
    }
    __syncthreads();
    float t = s_run[threadIdx.x];
    for (uint32_t b = b0; b < b0 + per && b < nt; b++) {
        tile_off[b] = t;
        t += tile_sum[b];
    }
}

// Batch row j <- the record whose cumulative-weight interval holds
// (j + u) / B of the total (first r with G(r) > t, G the inclusive prefix
// sum, G(r) = tile_off[r / tile] + w_scanned[r]).
__global__ void k_resample(const float* __restrict__ rec, uint32_t R, const float* __restrict__ cdf,
                           const float* __restrict__ tile_off, uint32_t nt, uint32_t B, float u,
                           float* __restrict__ x, float* __restrict__ d, float* __restrict__ c) {
    const float total = tile_off[nt];
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < B; j += gridDim.x * blockDim.x) {
        if (!(total > 0.0f) || !isfinite(total)) {
            write_batch_row(rec, 0.0f, j, x, d, c);
            continue;
        }
        const float t = ((float)j + u) * (total / (float)B);
        uint32_t lo = 0, hi = R;  // first r in [lo, hi) with G(r) > t, or R
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            const float g = tile_off[mid / kScanTile] + cdf[mid];
            if (g > t)
                hi = mid;
            else
                lo = mid + 1;
        }
        const uint32_t r = lo < R ? lo : R - 1;
        const float g_prev = r == 0 ? 0.0f : tile_off[(r - 1) / kScanTile] + cdf[r - 1];
        const float g_r = tile_off[r / kScanTile] + cdf[r];
        write_batch_row(rec + (size_t)r * kGRecFloats, g_r > g_prev ? 1.0f : 0.0f, j, x, d, c);
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// the device bytes the render service reserves for a guided render
static_assert(kGuideBatch == dl_sizes::kGuideBatchRows && kScanTile == (int)dl_sizes::kGuideScanTile && kGParams == dl_sizes::kGuideParams &&
                  kGWSlot == dl_sizes::kGuideWSlot,
              "guided render sizes");
static_assert(dl_sizes::kGuideNetBytes == 4ull * kGParams * sizeof(float) + 5 * 64 * sizeof(float) +
                                              3ull * 5 * kGWSlot * sizeof(uint16_t) +
                                              (1 + kSumBlocks + dl_sizes::kGuideTrainBlocks) * sizeof(float),
              "guide_init allocations");
static_assert(dl_sizes::kGuideTrainBytes == (uint64_t)kGuideBatch * (kGIn + 3 + 1) * sizeof(float) +
                                                (uint64_t)dl_sizes::kGuideTrainBlocks * kGParams * sizeof(float),
              "training batch and partial gradients");

struct GuideState {
    // training batch built from render records
    uint32_t batch_cap = 0;
    float *bx = nullptr, *bd = nullptr, *bc = nullptr;
    // record weights (prefix-summed in place) and their tile offsets
    uint32_t rw_cap = 0;
    float *rw = nullptr, *tile_sum = nullptr, *tile_off = nullptr;
    float *theta = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr, *bias = nullptr;
    uint16_t *w = nullptr, *w16 = nullptr, *wt16 = nullptr;
    int step = 0;
    float lr = 1e-2f;
    float* scalars = nullptr;  // the step's loss, the partial sums of the weights, the blocks' losses
    float* part = nullptr;     // per-block partial gradients of a training step
    std::vector<void*> allocs;
};

namespace {

template <typename T>
dl_status galloc(Ctx* c, GuideState* g, T** p, size_t count) {
    void* q = nullptr;
    DL_HIP_CHECK(c, dmalloc(c, &q, std::max<size_t>(1, count) * sizeof(T)));
    g->allocs.push_back(q);
    *p = (T*)q;
    return DL_OK;
}

#define DL_TRY(expr)                \
    do {                            \
        dl_status s_ = (expr);      \
        if (s_ != DL_OK) return s_; \
    } while (0)

Net net_of(const GuideState* g) { return Net{g->w, g->w16, g->wt16, g->bias}; }

// Deterministic initial weights: He-uniform (last layer x0.1), zero biases,
// uniforms from splitmix64 (Steele et al. 2014).
void init_weights(uint64_t seed, std::vector<float>& th) {
    th.assign(kGParams, 0.0f);
    uint64_t x = seed;
    auto next = [&x]() {
        uint64_t z = (x += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (float)((z >> 40) * (1.0 / 16777216.0));
    };
    for (int l = 0; l < 5; l++) {
        const float a = std::sqrt(6.0f / glayer_in(l)) * (l == 4 ? 0.1f : 1.0f);
        for (int k = 0; k < glayer_out(l) * glayer_in(l); k++) th[glayer_w(l) + k] = (2.0f * next() - 1.0f) * a;
    }
}

}  // namespace

void free_guide(Ctx* c) {
    GuideState* g = (GuideState*)c->guide;
    if (!g) return;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    for (void* p : g->allocs) (void)dfree(c, p);
    delete g;
    c->guide = nullptr;
}

dl_status guide_init(Ctx* c, uint64_t seed, float lr, const float* params) {
    free_guide(c);
    GuideState* g = new GuideState();
    c->guide = g;
    g->lr = lr;
    DL_TRY(galloc(c, g, &g->theta, kGParams));
    DL_TRY(galloc(c, g, &g->m, kGParams));
    DL_TRY(galloc(c, g, &g->v, kGParams));
    DL_TRY(galloc(c, g, &g->grad, kGParams));
    DL_TRY(galloc(c, g, &g->bias, 5 * 64));
    DL_TRY(galloc(c, g, &g->w, 5 * kGWSlot));
    DL_TRY(galloc(c, g, &g->w16, 5 * kGWSlot));
    DL_TRY(galloc(c, g, &g->wt16, 5 * kGWSlot));
    DL_TRY(galloc(c, g, &g->scalars, 1 + kSumBlocks + dl_sizes::kGuideTrainBlocks));
    std::vector<float> th;
    if (params)
        th.assign(params, params + kGParams);
    else
        init_weights(seed, th);
    DL_HIP_CHECK(c, hipMemcpyAsync(g->theta, th.data(), kGParams * sizeof(float), hipMemcpyHostToDevice, c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->m, 0, kGParams * sizeof(float), c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->v, 0, kGParams * sizeof(float), c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->grad, 0, kGParams * sizeof(float), c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->w, 0, 5 * kGWSlot * sizeof(uint16_t), c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->w16, 0, 5 * kGWSlot * sizeof(uint16_t), c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->wt16, 0, 5 * kGWSlot * sizeof(uint16_t), c->stream));
    DL_HIP_CHECK(c, hipMemsetAsync(g->bias, 0, 5 * 64 * sizeof(float), c->stream));
    k_refresh<<<(kGParams + 255) / 256, 256, 0, c->stream>>>(g->theta, g->w, g->w16, g->wt16, g->bias);
    DL_HIP_CHECK(c, hipGetLastError());
    return DL_OK;
}

// Forward pass over n float32 input rows (device), raw outputs to out.
dl_status guide_forward(Ctx* c, const float* x, uint32_t n, float* out) {
    GuideState* g = (GuideState*)c->guide;
    if (n == 0) return DL_OK;
    const uint32_t tiles = (n + kGRowsPerWave - 1) / kGRowsPerWave;
    const int grid = (int)std::max<uint32_t>(1, std::min<uint32_t>((tiles + kGWaves - 1) / kGWaves, (uint32_t)c->num_cus * 4));
    k_mlp_forward<<<grid, kGWaves * 64, 0, c->stream>>>(net_of(g), x, n, out);
    DL_HIP_CHECK(c, hipGetLastError());
    return DL_OK;
}

// One training step on n records (device arrays): gradient, then Adam.
dl_status guide_train(Ctx* c, const float* x, const float* dirs, const float* cw, uint32_t n, bool apply) {
    GuideState* g = (GuideState*)c->guide;
    if (!g->part) DL_TRY(galloc(c, g, &g->part, (size_t)dl_sizes::kGuideTrainBlocks * kGParams));
    const uint32_t blocks = dl_sizes::guide_train_blocks(n);
    float* const sums = g->scalars + 1;
    float* const losses = sums + kSumBlocks;
    k_sum<<<kSumBlocks, 256, 0, c->stream>>>(cw, n, sums);
    k_train<<<blocks, kTrainWaves * 64, 0, c->stream>>>(net_of(g), x, dirs, cw, n, sums, g->part, losses);
    if (apply) g->step++;
    AdamArgs a{g->theta, g->m, g->v, g->grad, g->lr, 1.0f - std::pow(0.9f, (float)g->step),
               1.0f - std::pow(0.999f, (float)g->step), apply ? 1 : 0, g->w, g->w16, g->wt16, g->bias};
    k_train_reduce<<<(kGParams + 63) / 64, 256, 0, c->stream>>>(g->part, blocks, a, losses, g->scalars);
    DL_HIP_CHECK(c, hipGetLastError());
    return DL_OK;
}

int guide_step_count(Ctx* c) { return c->guide ? ((GuideState*)c->guide)->step : 0; }

Net guide_net(Ctx* c) { return net_of((GuideState*)c->guide); }

// `steps` Adam steps on batches of kGuideBatch records resampled from the R
// render records in proportion to their weights; returns the steps taken.
dl_status guide_train_records(Ctx* c, const float* records, uint32_t R, const float4* rad, int steps) {
    GuideState* g = (GuideState*)c->guide;
    if (R == 0 || steps <= 0) return DL_OK;
    const uint32_t B = kGuideBatch;
    if (g->batch_cap < B) {
        for (float** p : {&g->bx, &g->bd, &g->bc})
            if (*p) {
                dfree(c, *p);
                g->allocs.erase(std::find(g->allocs.begin(), g->allocs.end(), (void*)*p));
            }
        g->batch_cap = B;
        DL_TRY(galloc(c, g, &g->bx, (size_t)B * kGIn));
        DL_TRY(galloc(c, g, &g->bd, (size_t)B * 3));
        DL_TRY(galloc(c, g, &g->bc, B));
    }
    const uint32_t nt = (R + kScanTile - 1) / kScanTile;
    if (g->rw_cap < R) {
        for (float** p : {&g->rw, &g->tile_sum, &g->tile_off})
            if (*p) {
                dfree(c, *p);
                g->allocs.erase(std::find(g->allocs.begin(), g->allocs.end(), (void*)*p));
            }
        g->rw_cap = R;
        DL_TRY(galloc(c, g, &g->rw, R));
        DL_TRY(galloc(c, g, &g->tile_sum, nt));
        DL_TRY(galloc(c, g, &g->tile_off, nt + 1));
    }
    const int eg = std::max(1, std::min<int>((int)((R + 255) / 256), c->num_cus * 8));
    // weights, their total, then the capped weights and their prefix sums
    k_record_weights<<<eg, 256, 0, c->stream>>>(records, R, rad, nullptr, 0.0f, g->rw);
    k_scan_tiles<<<nt, kScanThreads, 0, c->stream>>>(g->rw, R, g->tile_sum);
    k_scan_top<<<1, kScanThreads, 0, c->stream>>>(g->tile_sum, nt, g->tile_off);
    k_record_weights<<<eg, 256, 0, c->stream>>>(records, R, rad, g->tile_off + nt, kGuideMaxShare, g->rw);
    k_scan_tiles<<<nt, kScanThreads, 0, c->stream>>>(g->rw, R, g->tile_sum);
    k_scan_top<<<1, kScanThreads, 0, c->stream>>>(g->tile_sum, nt, g->tile_off);
    DL_HIP_CHECK(c, hipGetLastError());
    const int bg = std::max(1, std::min<int>((int)((B + 255) / 256), c->num_cus * 8));
    for (int s = 0; s < steps; s++) {
        // stratum offset of this step: golden-ratio sequence over the steps
        const double u = std::fmod(0.5 + 0.6180339887498949 * (double)(g->step + 1), 1.0);
        k_resample<<<bg, 256, 0, c->stream>>>(records, R, g->rw, g->tile_off, nt, B, (float)u, g->bx, g->bd, g->bc);
        DL_HIP_CHECK(c, hipGetLastError());
        DL_TRY(guide_train(c, g->bx, g->bd, g->bc, B, true));
    }
    return DL_OK;
}

dl_status guide_decode_rows(Ctx* c, const float* out, uint32_t n, float* mix) {
    if (n == 0) return DL_OK;
    k_mlp_decode<<<std::max(1, std::min<int>((int)((n + 255) / 256), c->num_cus * 8)), 256, 0, c->stream>>>(out, n,
                                                                                                        mix);
    DL_HIP_CHECK(c, hipGetLastError());
    return DL_OK;
}

}  // namespace dl

using namespace dl;

extern "C" {

dl_status dl_hip_guide_init(void* h, uint64_t seed, float lr, const float* params) {
    Ctx* c = (Ctx*)h;
    if (!c) return DL_ERR_INVALID;
    (void)hipSetDevice(c->device);
    return guide_init(c, seed, lr, params);
}

dl_status dl_hip_guide_params(void* h, float* params, float* grads) {
    Ctx* c = (Ctx*)h;
    if (!c) return DL_ERR_INVALID;
    GuideState* g = (GuideState*)c->guide;
    if (!g) return set_error(c, DL_ERR_STATE, "guide not initialised");
    (void)hipSetDevice(c->device);
    if (params)
        DL_HIP_CHECK(c, hipMemcpyAsync(params, g->theta, kGParams * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    if (grads)
        DL_HIP_CHECK(c, hipMemcpyAsync(grads, g->grad, kGParams * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    return DL_OK;
}

dl_status dl_hip_guide_eval(void* h, const float* x, uint32_t n, float* out, float* mix) {
    Ctx* c = (Ctx*)h;
    if (!c || !x || !out) return DL_ERR_INVALID;
    if (!c->guide) return set_error(c, DL_ERR_STATE, "guide not initialised");
    (void)hipSetDevice(c->device);
    DL_TRY(guide_forward(c, x, n, out));
    if (mix) DL_TRY(guide_decode_rows(c, out, n, mix));
    DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    return DL_OK;
}

dl_status dl_hip_guide_train_step(void* h, const float* x, const float* dirs, const float* weights, uint32_t n,
                                  int apply, float* loss) {
    Ctx* c = (Ctx*)h;
    if (!c || !x || !dirs || !weights) return DL_ERR_INVALID;
    GuideState* g = (GuideState*)c->guide;
    if (!g) return set_error(c, DL_ERR_STATE, "guide not initialised");
    if (n == 0) return set_error(c, DL_ERR_INVALID, "empty batch");
    (void)hipSetDevice(c->device);
    DL_TRY(guide_train(c, x, dirs, weights, n, apply != 0));
    if (loss) DL_HIP_CHECK(c, hipMemcpyAsync(loss, g->scalars, sizeof(float), hipMemcpyDeviceToHost, c->stream));
    DL_HIP_CHECK(c, hipStreamSynchronize(c->stream));
    return DL_OK;
}

}  // extern "C"
