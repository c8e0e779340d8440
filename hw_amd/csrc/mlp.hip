// mlp.hip -- the learned initialiser of the EM: a 128 -> 256 -> 256 -> 11
// perceptron with ReLU hidden layers, inference and training on the matrix
// cores (bfloat16 operands, fp32 accumulation).  No reference counterpart.
//
// Parameter vector (fp32 master copy, PyTorch Linear convention W[out][in]):
//   W1[256][128] b1[256] W2[256][256] b2[256] W3[11][256] b3[11]
// A bf16 mirror of the whole vector feeds the matrix cores; biases are added
// in fp32 from the master copy.
//
// Every product is v_mfma_f32_32x32x16_bf16 over k in steps of 16.  Operand lanes: lane l
// supplies A[l%32][k0+8(l/32)+j] and B[k0+8(l/32)+j][l%32], j = 0..7; the 16
// accumulators of lane l hold C[8(i/4)+4(l/32)+i%4][l%32].

#include "internal.h"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

namespace hwpa {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int MI = HWPA_MLP_IN, MH = HWPA_MLP_HIDDEN, MO = HWPA_MLP_OUT;
constexpr size_t OFF_W1 = 0;
constexpr size_t OFF_B1 = OFF_W1 + (size_t)MH * MI;
constexpr size_t OFF_W2 = OFF_B1 + MH;
constexpr size_t OFF_B2 = OFF_W2 + (size_t)MH * MH;
constexpr size_t OFF_W3 = OFF_B2 + MH;
constexpr size_t OFF_B3 = OFF_W3 + (size_t)MO * MH;
constexpr size_t NPARAM = OFF_B3 + MO;
static_assert(NPARAM == HWPA_MLP_PARAMS, "parameter count");

__device__ __forceinline__ bool PositiveBf16(uint16_t b) { return b != 0 && (b & 0x8000u) == 0; }

__device__ __forceinline__ bf16x8 LoadRow8(const uint16_t* __restrict__ p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}

// ---- features: 300-bin lane histogram -> 128 re-binned, normalised bf16 ----
// x[i] = 16 * (cnt[2i] + cnt[2i+1]) / N,  N = sum of cnt[0..255] (x = 0 if N = 0).
__global__ __launch_bounds__(64) void FeaturesKernel(const hwpa_lane_hist* __restrict__ hists, uint16_t* __restrict__ x)
{
    const int lane = blockIdx.x, z = threadIdx.x;
    const hwpa_lane_hist& h = hists[lane];
    uint32_t total = 0;
    for (int b = 0; b < 2 * MI; ++b) total += h.bin_count[b][z];
    const float scale = total ? 16.0f / (float)total : 0.0f;
    uint4* out = reinterpret_cast<uint4*>(x + ((size_t)lane * LS + z) * MI);
    for (int i = 0; i < MI; i += 8) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b0 = 2 * (i + 2 * j), b1 = b0 + 2;
            const float v0 = (float)(h.bin_count[b0][z] + h.bin_count[b0 + 1][z]) * scale;
            const float v1 = (float)(h.bin_count[b1][z] + h.bin_count[b1 + 1][z]) * scale;
            w[j] = (uint32_t)hw_f2bf(v0) | ((uint32_t)hw_f2bf(v1) << 16);
        }
        out[i / 8] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// ---- training targets from the EM diagnostics ---------------------------------
// Raw units: u = 2 * binSize (one re-binned bin), origin at the histogram's
// lower bound:  r0 = (mu_bl - lo) / u,  r1 = log(var_bl / u^2),
// r2..5 = (mu_a - lo) / u,  r6..10 = mixture weights (softmax targets),
// r11 = 1 when the estimate is a valid target (converged, status OK, enough
// confidence), else 0 (the confidence output's target).
__global__ __launch_bounds__(64) void TargetsKernel(const hwpa_lane_hist* __restrict__ hists,
                                                    const float* __restrict__ diag, float minConf,
                                                    float* __restrict__ t, uint8_t* __restrict__ valid)
{
    const int lane = blockIdx.x, z = threadIdx.x;
    const float* dg = diag + (size_t)lane * HWPA_EM_DIAG_ROWS * LS + z;
    const float lo = hists[lane].low_bound[z], u = 2.0f * hists[lane].bin_size[z];
    float* o = t + ((size_t)lane * LS + z) * MO;
    const float var0 = dg[(10 + 0) * LS];
    o[0] = (dg[(5 + 0) * LS] - lo) / u;
    o[1] = hw_logf(var0 / (u * u));
    for (int a = 0; a < NA; ++a) o[2 + a] = (dg[(5 + 1 + a) * LS] - lo) / u;
    for (int k = 0; k < 5; ++k) o[6 + k] = dg[k * LS];
    const bool ok = dg[16 * LS] > 0.0f && dg[17 * LS] == 0.0f && dg[15 * LS] >= minConf &&
                    hw_isfinite(o[0]) && hw_isfinite(o[1]) && var0 > 0.0f;
    o[11] = ok ? 1.0f : 0.0f;
    valid[(size_t)lane * LS + z] = ok ? 1 : 0;
}

// ---- loss ----------------------------------------------------------------------
// Network output j < 6 stands for the raw target off[j] + scale[j] * y[j]; the
// loss is sum_j w[j] (y[j] - (r[j] - off[j]) / scale[j])^2 + w[6] * CE(softmax(y[6..10]), r[6..10])
// + w[7] * BCE(sigmoid(y[11]), r[11]), the last as softplus(y) - r y in its stable form
// max(y, 0) - r y + log(1 + exp(-|y|)).  Samples marked invalid keep only the last term.
// omap = {off[6], scale[6], w[8]}.
// One sample: its loss and the gradient g of the batch's mean loss with respect to y.
__device__ __forceinline__ float SampleLoss(const float* yb, const float* tb, bool valid, float invB, const float* omap,
                                            float (&g)[MO])
{
    // Confidence output: logistic loss against target 11.
    const float wg = omap[19];
    const float yc = yb[11], tc = tb[11];
    const float ez = hw_expf(-hw_fabsf(yc));
    float loss = wg * ((hw_maxf(yc, 0.0f) - tc * yc) + hw_logf(1.0f + ez));
    const float sg = (yc >= 0.0f) ? 1.0f / (1.0f + ez) : ez / (1.0f + ez);
    g[11] = (wg * (sg - tc)) * invB;
    if (!valid) {
#pragma unroll
        for (int j = 0; j < 11; ++j) g[j] = 0.0f;
        return loss;
    }
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const float tn = (tb[j] - omap[j]) / omap[6 + j];
        const float d = yb[j] - tn;
        const float w = omap[12 + j];
        loss += w * (d * d);
        g[j] = ((2.0f * w) * d) * invB;
    }
    const float wce = omap[18];
    float mx = yb[6];
    for (int k = 1; k < 5; ++k) mx = hw_maxf(mx, yb[6 + k]);
    float e[5], se = 0.0f;
    for (int k = 0; k < 5; ++k) {
        e[k] = hw_expf(yb[6 + k] - mx);
        se += e[k];
    }
    const float lse = mx + hw_logf(se);
    for (int k = 0; k < 5; ++k) {
        const float p = e[k] / se;
        loss -= wce * (tb[6 + k] * (yb[6 + k] - lse));
        g[6 + k] = (wce * (p - tb[6 + k])) * invB;
    }
    return loss;
}

// ---- training ------------------------------------------------------------------
// A step is two launches: TrainRowsKernel takes every row through the forward pass, the loss and
// the gradients of its hidden units, TrainGradKernel sums the weight gradients over the batch and
// takes the Adam step.
//
// Between them the matrices lie as the batch-long products read them, [block of 16 rows][unit][16
// rows], the 16 in the order in which the accumulators of a 32x32 product hold them (the halves
// of a wave: rows 0-3, 8-11 and 4-7, 12-15): a lane's accumulators are two 16-byte stores, and an
// operand of a k-step is one contiguous KB.  Any order serves a sum over the batch as long as all
// matrices share it.
constexpr int kTrainRows = 32;             // rows of a TrainRowsKernel workgroup
constexpr int kTrainWaves = MH / 32;       // one wave per 32 hidden units
constexpr int kGradWaves = 16;
constexpr int kGradTiles2 = (MH / 32) * (MH / 32), kGradTiles1 = (MH / 32) * (MI / 32), kGradTiles3 = MH / 32;
constexpr int kGradTiles = kGradTiles2 + kGradTiles1 + kGradTiles3;
constexpr int kOutPad = 16;                // outputs padded to one k-step
constexpr int kPart = MO + 1;              // per 32 rows: sums of dY's columns, sum of the losses

// Training buffers, sized for whole 32-row blocks.
struct TrainActs {
    uint16_t *X, *H1, *H2, *dH1, *dH2, *dY;
    float* part;
};

struct AdamArgs {
    float *P, *Mo, *Ve;
    uint16_t *Pb, *WT;
    float lr, b1, b2, c1, c2, eps;
};

// bf16 mirrors of the weights in operand order, [16-wide k-step][unit][16 k], so that a wave reads a
// k-step of 32 units as one KB: W1, W2, and transposed W2 and W3 (its k-step padded with zeros).
constexpr size_t OFF_O1 = 0;
constexpr size_t OFF_O2 = OFF_O1 + (size_t)MH * MI;
constexpr size_t OFF_T2 = OFF_O2 + (size_t)MH * MH;
constexpr size_t OFF_T3 = OFF_T2 + (size_t)MH * MH;
constexpr size_t NTRANS = OFF_T3 + (size_t)MH * kOutPad;

__device__ __forceinline__ uint32_t OperandAt(uint32_t unit, uint32_t k) { return ((k >> 4) * MH + unit) * 16 + (k & 15); }

// Parameter i into the bf16 mirrors.
__device__ __forceinline__ void StoreBf16(uint32_t i, float v, uint16_t* __restrict__ pb, uint16_t* __restrict__ wt)
{
    const uint16_t h = hw_f2bf(v);
    pb[i] = h;
    if (i < OFF_B1) {
        wt[OFF_O1 + OperandAt(i / MI, i % MI)] = h;
    } else if (i >= OFF_W2 && i < OFF_B2) {
        const uint32_t e = i - (uint32_t)OFF_W2;
        wt[OFF_O2 + OperandAt(e / MH, e % MH)] = h;
        wt[OFF_T2 + OperandAt(e % MH, e / MH)] = h;
    } else if (i >= OFF_W3 && i < OFF_B3) {
        const uint32_t e = i - (uint32_t)OFF_W3;
        wt[OFF_T3 + OperandAt(e % MH, e / MH)] = h;
    }
}

__global__ __launch_bounds__(256) void ToBf16Kernel(const float* __restrict__ p, uint16_t* __restrict__ pb,
                                                    uint16_t* __restrict__ wt, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) StoreBf16(i, p[i], pb, wt);
    if (i < MH * (kOutPad - MO)) wt[OFF_T3 + (size_t)(i / (kOutPad - MO)) * kOutPad + MO + i % (kOutPad - MO)] = 0;
}

// Forward, loss and hidden gradients of 32 rows per workgroup, one wave per 32 hidden units.  At a
// training batch the kernel is a chain of small products, so what bounds it is latency: every wave
// requests its share of the weights well before their products (8 + 16 + 16 k-steps, 40 KB, one
// contiguous KB each: read in the parameters' own order, 32 B of each line at a time, the kernel
// took 30 us), targets and output weights are staged with the inputs, the activations go from
// layer to layer in LDS, and the ReLU masks stay in registers.  Batch 4,096 (128 workgroups): 17
// us, where the forward pass (16 workgroups of 256 rows), the loss and two products with operands
// gathered 2 bytes at a time took 36 + 5 + 11 + 20 us.
__global__ __launch_bounds__(64 * kTrainWaves) void TrainRowsKernel(const uint16_t* __restrict__ x,
                                                                    const float* __restrict__ t,
                                                                    const uint8_t* __restrict__ valid, uint32_t batch,
                                                                    const uint16_t* __restrict__ Wb,
                                                                    const uint16_t* __restrict__ WT,
                                                                    const float* __restrict__ P,
                                                                    const float* __restrict__ omap, TrainActs w)
{
    constexpr int kXs = MI + 8, kHs = MH + 8, kYs = 24;
    __shared__ __align__(16) uint16_t xs[kTrainRows][kXs];
    __shared__ __align__(16) uint16_t hs[3][kTrainRows][kHs];   // h1, h2, dh2
    __shared__ __align__(16) uint16_t dys[kTrainRows][kYs];
    __shared__ __align__(16) uint16_t w3s[MO][kHs];
    __shared__ float ys[kTrainRows][MO + 1], dyf[kTrainRows][kPart], ts[kTrainRows][MO + 1], om[20];
    __shared__ uint8_t vs[kTrainRows];
    static_assert(64 * kTrainWaves == kTrainRows * MI / 8, "one 16-byte piece of the inputs per thread");
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, r = l & 31, half = l >> 5, kq = half * 8;
    const int n = wave * 32 + r;   // this lane's hidden unit
    bf16x8 w1[MI / 16], w2[MH / 16], wt[MH / 16];
#pragma unroll
    for (int k = 0; k < MI / 16; ++k) w1[k] = LoadRow8(WT + OFF_O1 + ((size_t)k * MH + n) * 16 + kq);
#pragma unroll
    for (int k = 0; k < MH / 16; ++k) w2[k] = LoadRow8(WT + OFF_O2 + ((size_t)k * MH + n) * 16 + kq);
    const bf16x8 w3t = LoadRow8(WT + OFF_T3 + (size_t)n * kOutPad + kq);
    const float b1 = P[OFF_B1 + n], b2 = P[OFF_B2 + n], b3 = P[OFF_B3 + (r < MO ? r : 0)];
    const float invB = 1.0f / (float)batch;
    auto rowOf = [&](int i) { return (i >> 2) * 8 + half * 4 + (i & 3); };
    auto pack = [](uint32_t lo, uint32_t hi) { return lo | (hi << 16); };
    const uint32_t blk = blockIdx.x;
    const uint32_t m0 = blk * kTrainRows;
    const uint32_t live = min(batch - m0, (uint32_t)kTrainRows);
    // A lane's 16 values of one unit: two pieces of the batch-long layout.
    auto storeUnits = [&](uint16_t* base, const uint32_t (&v)[8]) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            *reinterpret_cast<uint4*>(base + ((((size_t)blk * 2 + q) * MH + n) * 2 + half) * 8) =
                make_uint4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    };
    auto storeRows = [&](uint16_t (*h)[kHs], const uint32_t (&v)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            h[rowOf(2 * i)][n] = (uint16_t)v[i];
            h[rowOf(2 * i + 1)][n] = (uint16_t)(v[i] >> 16);
        }
    };
    // Rows past the batch are zero throughout.
    {
        const int row = threadIdx.x >> 4, c = (threadIdx.x & 15) * 8;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if ((uint32_t)row < live) v = *reinterpret_cast<const uint4*>(x + (size_t)(m0 + row) * MI + c);
        float tv = 0.0f;
        uint4 wv = make_uint4(0u, 0u, 0u, 0u);
        static_assert(kTrainRows * MO <= 64 * kTrainWaves && MO * MH / 8 <= 64 * kTrainWaves, "one load per thread");
        if (threadIdx.x < live * MO) tv = t[(size_t)m0 * MO + threadIdx.x];
        if (threadIdx.x < MO * MH / 8) wv = *reinterpret_cast<const uint4*>(Wb + OFF_W3 + (size_t)threadIdx.x * 8);
        if (threadIdx.x < 20) om[threadIdx.x] = omap[threadIdx.x];
        if (threadIdx.x < live) vs[threadIdx.x] = !valid || valid[m0 + threadIdx.x] != 0;
        *reinterpret_cast<uint4*>(&xs[row][c]) = v;
        if (threadIdx.x < kTrainRows * MO) ts[threadIdx.x / MO][threadIdx.x % MO] = tv;
        if (threadIdx.x < MO * MH / 8)
            *reinterpret_cast<uint4*>(&w3s[threadIdx.x / (MH / 8)][threadIdx.x % (MH / 8) * 8]) = wv;
    }
    __syncthreads();
    {
        const int q = threadIdx.x >> 8, f = (threadIdx.x >> 1) & (MI - 1), hf = threadIdx.x & 1;
        uint32_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = q * 16 + (j >> 1) * 8 + hf * 4 + (j & 1) * 2;
            v[j] = pack(xs[row][f], xs[row + 1][f]);
        }
        *reinterpret_cast<uint4*>(w.X + ((((size_t)blk * 2 + q) * MI + f) * 2 + hf) * 8) =
            make_uint4(v[0], v[1], v[2], v[3]);
    }
    f32x16 acc{};
#pragma unroll
    for (int k = 0; k < MI / 16; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(LoadRow8(&xs[r][16 * k + kq]), w1[k], acc, 0, 0, 0);
    auto relu = [&](float b, uint32_t (&v)[8]) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float z = acc[i] + b;
            uint32_t h = hw_f2bf_nonnan(z > 0.0f ? z : 0.0f);
            if ((uint32_t)rowOf(i) >= live) h = 0;
            v[i >> 1] = (i & 1) ? pack(v[i >> 1], h) : h;
        }
    };
    auto masked = [&](const uint32_t (&h)[8], uint32_t (&v)[8]) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint32_t d =
                PositiveBf16((uint16_t)(h[i >> 1] >> (16 * (i & 1)))) ? (uint32_t)hw_f2bf(acc[i]) : 0u;
            v[i >> 1] = (i & 1) ? pack(v[i >> 1], d) : d;
        }
    };
#pragma unroll
    for (int k = 0; k < MH / 16; ++k) wt[k] = LoadRow8(WT + OFF_T2 + ((size_t)k * MH + n) * 16 + kq);
    uint32_t h1[8], h2[8], d[8];
    relu(b1, h1);
    storeRows(hs[0], h1);
    storeUnits(w.H1, h1);
    __syncthreads();
    acc = f32x16{};
#pragma unroll
    for (int k = 0; k < MH / 16; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(LoadRow8(&hs[0][r][16 * k + kq]), w2[k], acc, 0, 0, 0);
    relu(b2, h2);
    storeRows(hs[1], h2);
    storeUnits(w.H2, h2);
    __syncthreads();
    if (wave == 0) {
        // Outputs: one 32-column product of which MO columns are real.
        const bf16x8 zero8 = __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u));
        acc = f32x16{};
#pragma unroll
        for (int k = 0; k < MH / 16; ++k) {
            const bf16x8 w3 = r < MO ? LoadRow8(&w3s[r][16 * k + kq]) : zero8;
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(LoadRow8(&hs[1][r][16 * k + kq]), w3, acc, 0, 0, 0);
        }
        if (r < MO) {
#pragma unroll
            for (int i = 0; i < 16; ++i) ys[rowOf(i)][r] = acc[i] + b3;
        }
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)kTrainRows) {
        float g[MO] = {}, loss = 0.0f;
        if (threadIdx.x < live) {
            loss = SampleLoss(ys[threadIdx.x], ts[threadIdx.x], vs[threadIdx.x] != 0, invB, om, g);
        }
#pragma unroll
        for (int j = 0; j < kOutPad; ++j) dys[threadIdx.x][j] = j < MO ? hw_f2bf(g[j < MO ? j : 0]) : (uint16_t)0;
#pragma unroll
        for (int j = 0; j < MO; ++j) dyf[threadIdx.x][j] = g[j];
        dyf[threadIdx.x][MO] = loss;
    }
    __syncthreads();
    if (threadIdx.x < kPart) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < kTrainRows; ++i) s += dyf[i][threadIdx.x];
        w.part[(size_t)blk * kPart + threadIdx.x] = s;
    } else if (wave == 1) {
        const int q = l >> 5, o = (l >> 1) & (kOutPad - 1), hf = l & 1;
        uint32_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = q * 16 + (j >> 1) * 8 + hf * 4 + (j & 1) * 2;
            v[j] = pack(dys[row][o], dys[row + 1][o]);
        }
        *reinterpret_cast<uint4*>(w.dY + ((((size_t)blk * 2 + q) * kOutPad + o) * 2 + hf) * 8) =
            make_uint4(v[0], v[1], v[2], v[3]);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(LoadRow8(&dys[r][kq]), w3t, f32x16{}, 0, 0, 0);
    masked(h2, d);
    storeRows(hs[2], d);
    storeUnits(w.dH2, d);
    __syncthreads();
    acc = f32x16{};
#pragma unroll
    for (int k = 0; k < MH / 16; ++k)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(LoadRow8(&hs[2][r][16 * k + kq]), wt[k], acc, 0, 0, 0);
    masked(h1, d);
    storeUnits(w.dH1, d);
}

__device__ __forceinline__ void AdamOne(uint32_t i, float gi, float p0, float m0, float v0, const AdamArgs& a)
{
    const float mi = a.b1 * m0 + (1.0f - a.b1) * gi;
    const float vi = a.b2 * v0 + (1.0f - a.b2) * (gi * gi);
    a.Mo[i] = mi;
    a.Ve[i] = vi;
    const float mh = mi / a.c1, vh = vi / a.c2;
    const float pi = p0 - a.lr * mh / (hw_sqrtf(vh) + a.eps);
    a.P[i] = pi;
    StoreBf16(i, pi, a.Pb, a.WT);
}

// Weight gradients: one workgroup per 32x32 tile of W1, W2 and W3, its 16 waves taking every 16th
// 16-row block of the batch, their accumulators added in wave order through LDS; the bias gradients of
// W1 and W2 are one more product, with ones, of the tiles in the first column; the last workgroup
// adds the per-block sums of the outputs' gradients and of the losses.  STEP applies the Adam
// step to the sums, else they go to G.  Bound by the operand reads: 512 KB a tile at batch 4,096,
// contiguous, from the L2s (consecutive workgroups, which lie on different XCDs, differ in the
// tile's rows, so an XCD reads one eighth of one operand).  9 us there (10 with the step); split over
// the batch into 32 slices with operands gathered 2 bytes at a time, the three products took 65 us,
// the sums of the slices 27, of the columns 36 and of the losses 6, the Adam step 4.
template <bool STEP>
__global__ __launch_bounds__(64 * kGradWaves) void TrainGradKernel(TrainActs w, uint32_t batch, float* __restrict__ G,
                                                                   float* __restrict__ lossOut, AdamArgs a)
{
    __shared__ float red[kGradWaves][32 * 32];
    __shared__ float redB[kGradWaves][32];
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, r = l & 31, half = l >> 5;
    const uint32_t blocks = (batch + kTrainRows - 1) / kTrainRows;
    auto emit = [&](uint32_t i, float g, float p0, float m0, float v0) {
        if (STEP) AdamOne(i, g, p0, m0, v0, a);
        else G[i] = g;
    };
    int tile = (int)blockIdx.x;
    if (tile == kGradTiles) {
        static_assert(kPart <= kGradWaves, "one wave per sum");
        if (wave >= kPart) return;
        float s = 0.0f;
        for (uint32_t b = (uint32_t)l; b < blocks; b += 64) s += w.part[(size_t)b * kPart + wave];
        for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m, 64);
        if (l != 0) return;
        if (wave == MO) {
            *lossOut = s / (float)batch;
        } else {
            const uint32_t i = (uint32_t)OFF_B3 + (uint32_t)wave;
            if (STEP) emit(i, s, a.P[i], a.Mo[i], a.Ve[i]);
            else emit(i, s, 0.0f, 0.0f, 0.0f);
        }
        return;
    }
    const uint16_t *A, *B;
    int nfA = MH, nfB = MH, rows = 32, m0, n0;
    uint32_t off, offB = 0;
    bool bias = false;
    if (tile < kGradTiles2) {
        m0 = (tile % (MH / 32)) * 32;
        n0 = (tile / (MH / 32)) * 32;
        A = w.dH2;
        B = w.H1;
        off = (uint32_t)OFF_W2;
        offB = (uint32_t)OFF_B2;
        bias = n0 == 0;
    } else if (tile < kGradTiles2 + kGradTiles1) {
        tile -= kGradTiles2;
        m0 = (tile % (MH / 32)) * 32;
        n0 = (tile / (MH / 32)) * 32;
        A = w.dH1;
        B = w.X;
        nfB = MI;
        off = (uint32_t)OFF_W1;
        offB = (uint32_t)OFF_B1;
        bias = n0 == 0;
    } else {
        m0 = 0;
        n0 = (tile - kGradTiles2 - kGradTiles1) * 32;
        A = w.dY;
        B = w.H2;
        nfA = kOutPad;
        rows = MO;
        off = (uint32_t)OFF_W3;
    }
    // This thread's element of the tile, and its parameter's state in flight meanwhile.
    const int em = (wave >> 2) * 8 + half * 4 + (wave & 3), en = r;
    const uint32_t ei = off + (uint32_t)(m0 + em) * (uint32_t)nfB + (uint32_t)(n0 + en);
    const uint32_t bi = offB + (uint32_t)m0 + (uint32_t)r;
    const bool mine = em < rows, mineB = bias && threadIdx.x < 32;
    float p0 = 0.0f, mo = 0.0f, ve = 0.0f, pB = 0.0f, moB = 0.0f, veB = 0.0f;
    if (STEP && mine) {
        p0 = a.P[ei];
        mo = a.Mo[ei];
        ve = a.Ve[ei];
    }
    if (STEP && mineB) {
        pB = a.P[bi];
        moB = a.Mo[bi];
        veB = a.Ve[bi];
    }
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u));
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u));
    const uint32_t kb = blocks * 2;
    const bool aRow = r < nfA;
    const uint16_t* pa = A + ((size_t)(m0 + (aRow ? r : 0)) * 2 + half) * 8;
    const uint16_t* pb = B + ((size_t)(n0 + r) * 2 + half) * 8;
    const size_t sa = (size_t)nfA * 16, sb = (size_t)nfB * 16;
    f32x16 acc{}, accB{};
    constexpr uint32_t kDeep = 4;
    for (uint32_t k0 = (uint32_t)wave; k0 < kb; k0 += kGradWaves * kDeep) {
        bf16x8 va[kDeep], vb[kDeep];
#pragma unroll
        for (uint32_t j = 0; j < kDeep; ++j) {
            const uint32_t k = k0 + j * kGradWaves;
            va[j] = (aRow && k < kb) ? LoadRow8(pa + sa * k) : zero8;
            vb[j] = k < kb ? LoadRow8(pb + sb * k) : zero8;
        }
#pragma unroll
        for (uint32_t j = 0; j < kDeep; ++j) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[j], vb[j], acc, 0, 0, 0);
            if (bias) accB = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[j], ones, accB, 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) red[wave][i * 64 + l] = acc[i];
    if (bias && r == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) redB[wave][(i >> 2) * 8 + half * 4 + (i & 3)] = accB[i];
    }
    __syncthreads();
    float g = 0.0f;
#pragma unroll
    for (int k = 0; k < kGradWaves; ++k) g += red[k][threadIdx.x];
    if (mine) emit(ei, g, p0, mo, ve);
    if (mineB) {
        float gb = 0.0f;
#pragma unroll
        for (int k = 0; k < kGradWaves; ++k) gb += redB[k][r];
        emit(bi, gb, pB, moB, veB);
    }
}

}  // namespace hwpa

using namespace hwpa;

struct hwpa_initializer {
    float* P = nullptr;     // fp32 master parameters
    uint16_t* Pb = nullptr; // bf16 mirror
    float* G = nullptr;     // gradients
    float* Mo = nullptr;    // Adam moments
    float* Ve = nullptr;
    int64_t step = 0;
    uint16_t* WT = nullptr; // transposed bf16 mirrors (NTRANS)
    uint32_t batchCap = 0;  // rows the training buffers hold, whole 32-row blocks
    TrainActs acts{};
    float* lossDev = nullptr;
    float* omap = nullptr;      // device {off[6], scale[6], w[8]}
    float omapHost[20] = {};
    // A learned-start workspace kept between estimations (LearnedWsTake), at most one.
    std::mutex wsMutex;
    LearnedWs ws;
};

namespace hwpa {

// An estimation's workspace: the one the initialiser keeps if it is large enough, on the current
// device and not in use, else a new one.  Allocating and freeing its ten buffers on every call took
// 0.4 ms of a 4,096-lane estimation's 4.1.  A kept one that does not serve is freed first, so a
// call never needs more memory than its own workspace.
int32_t LearnedWsTake(hwpa_initializer* m, uint32_t lanes, LearnedWs& w)
{
    int device = -1;
    HWPA_HIP(hipGetDevice(&device));
    {
        std::lock_guard<std::mutex> g(m->wsMutex);
        std::swap(w, m->ws);
    }
    if (w.lanes >= lanes && w.device == device) return HWPA_OK;
    const int32_t rc = LearnedWsAlloc(w, lanes);   // (frees what w holds)
    w.device = device;
    return rc;
}

// Gives a workspace back once nothing uses it; the larger of it and the kept one stays (up to
// kKeepWsLanes lanes, 0.8 GB), the other is freed.
void LearnedWsGive(hwpa_initializer* m, LearnedWs& w)
{
    constexpr uint32_t kKeepWsLanes = 16384;
    if (w.lanes <= kKeepWsLanes) {
        std::lock_guard<std::mutex> g(m->wsMutex);
        if (w.lanes > m->ws.lanes) std::swap(w, m->ws);
    }
    LearnedWsFree(w);
}

static void FreeTrain(hwpa_initializer* m)
{
    DeviceFree(m->acts.X);
    DeviceFree(m->acts.H1);
    DeviceFree(m->acts.H2);
    DeviceFree(m->acts.dH1);
    DeviceFree(m->acts.dH2);
    DeviceFree(m->acts.dY);
    DeviceFree(m->acts.part);
    m->acts = TrainActs{};
    m->batchCap = 0;
}

static int32_t EnsureBatch(hwpa_initializer* m, uint32_t batch)
{
    if (batch <= m->batchCap) return HWPA_OK;
    // Buffers may still be in use by queued work on any stream.
    HWPA_HIP(hipDeviceSynchronize());
    FreeTrain(m);
    const size_t blocks = ((size_t)batch + kTrainRows - 1) / kTrainRows, rows = blocks * kTrainRows;
    TrainActs& w = m->acts;
    int32_t rc = DeviceAlloc((void**)&w.X, rows * MI * 2, "mlp activations");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&w.H1, rows * MH * 2, "mlp activations");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&w.H2, rows * MH * 2, "mlp activations");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&w.dH1, rows * MH * 2, "mlp gradients");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&w.dH2, rows * MH * 2, "mlp gradients");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&w.dY, rows * kOutPad * 2, "mlp gradients");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&w.part, blocks * kPart * 4, "mlp bias sums");
    if (rc != HWPA_OK) {
        FreeTrain(m);
        return rc;
    }
    m->batchCap = (uint32_t)std::min<size_t>(rows, UINT32_MAX);
    return HWPA_OK;
}

// Inference: 32 rows per wave, kFusedWaves (8) waves per workgroup.  Each layer is the
// 32x32x16 bf16 MFMA over 32-column tiles with k ascending, the arithmetic of the training
// kernels' forward pass; the hidden activations stay in LDS (row-major, read back as the next
// layer's operand).  The weights of each 16-wide k-step of layers 1 and 2 (all 256 output columns:
// 8 KB) are staged once per workgroup in LDS, double-buffered with one barrier per step, so
// the 8 waves (256 rows) of a workgroup share one read of them instead of each wave
// fetching all 192 KB from L2.
constexpr int kFusedRows = 32, kFusedWaves = 8, kHsStride = MH + 8;
constexpr int kSlab = MH * 16;   // bf16 weights of one k-step: [256 columns][16 k]

// HIST: the inputs are computed from the lane histograms as FeaturesKernel does (row =
// lane * 64 + ZMW), so inference reads the counters once and writes no input matrix.  Each
// half-wave needs half of the 128 re-binned inputs of its row (k-chunks kq = 0 / 8 of every
// 16-wide k-step): it sums exactly those bin pairs, the two halves' partial totals give the
// row total, and the scaled bf16 inputs stay in registers.
template <bool HIST>
__global__ __launch_bounds__(64 * kFusedWaves) void MlpFusedForwardKernel(const uint16_t* __restrict__ x,
                                                             const hwpa_lane_hist* __restrict__ hists, uint32_t rows,
                                                             const uint16_t* __restrict__ Wb,
                                                             const float* __restrict__ P, float* __restrict__ y)
{
    __shared__ __align__(16) uint16_t hs[kFusedWaves][kFusedRows][kHsStride];
    __shared__ __align__(16) uint16_t ws[2][kSlab];
    static_assert(64 * kFusedWaves == 2 * MH, "one 16-byte half column of a slab per thread");
    // 132 KiB of activations + 16 KiB of weight slabs: one workgroup per CU's 160 KiB of LDS.
    static_assert(sizeof(hs) + sizeof(ws) <= 160 * 1024, "LDS budget of a CU");
    // Thread t stages half t & 1 of column t >> 1 of a k-step's weights (16 bytes).
    const int sn = threadIdx.x >> 1, sh = (threadIdx.x & 1) * 8;
    auto slabLoad = [&](int off, int kdim, int k0) {
        return *reinterpret_cast<const uint4*>(Wb + off + (size_t)sn * kdim + k0 + sh);
    };
    auto slabStore = [&](int buf, uint4 v) { *reinterpret_cast<uint4*>(&ws[buf][sn * 16 + sh]) = v; };
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int r = l & 31, kq = (l >> 5) * 8;
    const int64_t m0 = ((int64_t)blockIdx.x * kFusedWaves + wave) * kFusedRows;
    const bool rowValid = m0 + r < (int64_t)rows;
    uint16_t (*h)[kHsStride] = hs[wave];
    auto hp = [&](int row, int col) { return &h[row][col]; };
    const bf16x8 zero8 = __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u));

    // Every product is (weights) x (activations): the weights are the A operand and a wave's 32
    // rows the B operand, so accumulator element i of lane l is output feature outRow(i) of
    // the tile (f32x16 layout of the 32x32 MFMA) for row r: each lane holds four runs of four
    // consecutive features of its own row.
    auto outRow = [&](int i) { return (i >> 2) * 8 + (l >> 5) * 4 + (i & 3); };
    // Bias, ReLU, bf16 and the row's activations back into LDS: one 8-byte store per run of four
    // features.
    auto hiddenOut = [&](const f32x16 (&a)[MH / 32], int boff) {
#pragma unroll
        for (int j = 0; j < MH / 32; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int f0 = j * 32 + g * 8 + (l >> 5) * 4;
                const float4 bias = *reinterpret_cast<const float4*>(P + boff + f0);
                const float bv[4] = {bias.x, bias.y, bias.z, bias.w};
                uint32_t hv[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float zv = a[j][4 * g + q] + bv[q];
                    hv[q] = hw_f2bf_nonnan(zv > 0.0f ? zv : 0.0f);
                }
                const uint2 pk = make_uint2(hv[0] | (hv[1] << 16), hv[2] | (hv[3] << 16));
                *reinterpret_cast<uint2*>(hp(r, f0)) = pk;
            }
        }
    };
    static_assert(OFF_B1 % 4 == 0 && OFF_B2 % 4 == 0 && (kHsStride * 2) % 8 == 0, "aligned runs of four");

    // ---- inputs from the histogram (HIST)
    uint32_t xin[MI / 16][4];
    if (HIST) {
        // The wave's 32 ZMWs x 2 MI bins of counters go through its activation buffer: 16-byte
        // loads of 8 ZMWs of one bin (a wave instruction moves 16 bins), then each lane reads
        // its ZMW's bins from LDS.  Rows come in whole half-lanes, so a wave is valid or not.
        static_assert(2 * MI * kFusedRows <= kFusedRows * kHsStride, "counters fit the activation buffer");
        uint16_t* hc = &h[0][0];   // [bin][32 ZMWs]
        if (m0 < (int64_t)rows) {
            const uint16_t* lb = &hists[m0 / LS].bin_count[0][m0 % LS];
            constexpr int NIT = 2 * MI / 16;
            const int piece = (l & 3) * 8;
            uint4 v[NIT];   // every load in flight before the first store
#pragma unroll
            for (int it = 0; it < NIT; ++it)
                v[it] = *reinterpret_cast<const uint4*>(lb + (size_t)(16 * it + (l >> 2)) * LS + piece);
#pragma unroll
            for (int it = 0; it < NIT; ++it)
                *reinterpret_cast<uint4*>(hc + (16 * it + (l >> 2)) * kFusedRows + piece) = v[it];
        }
        __syncthreads();
        uint32_t pair[MI / 16][8];
        uint32_t part = 0;
#pragma unroll
        for (int s = 0; s < MI / 16; ++s)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int i = 16 * s + kq + j;
                const uint32_t v =
                    rowValid ? (uint32_t)hc[(2 * i) * kFusedRows + r] + (uint32_t)hc[(2 * i + 1) * kFusedRows + r] : 0u;
                pair[s][j] = v;
                part += v;
            }
        const uint32_t total = part + (uint32_t)__shfl_xor((int)part, 32, 64);
        const float scale = total ? 16.0f / (float)total : 0.0f;
#pragma unroll
        for (int s = 0; s < MI / 16; ++s)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                xin[s][q] = (uint32_t)hw_f2bf_nonnan((float)pair[s][2 * q] * scale) |   // count x finite scale
                            ((uint32_t)hw_f2bf_nonnan((float)pair[s][2 * q + 1] * scale) << 16);
    }

    // ---- layer 1: [32 x MI] x [MI x MH]
    f32x16 acc[MH / 32];
#pragma unroll
    for (int j = 0; j < MH / 32; ++j) acc[j] = f32x16{};
    const uint16_t* xr = HIST ? nullptr : x + (m0 + r) * MI;
    // Weight slabs: step k + 1's slab is in flight during step k and stored after its
    // products; step k + 2's load is issued at the start of step k.
    uint4 next = slabLoad(OFF_W1, MI, 16);
    slabStore(0, slabLoad(OFF_W1, MI, 0));
    __syncthreads();
#pragma unroll
    for (int k0 = 0; k0 < MI; k0 += 16) {
        const int buf = (k0 / 16) & 1;
        uint4 next2{};
        if (k0 + 32 < MI) next2 = slabLoad(OFF_W1, MI, k0 + 32);
        bf16x8 a;
        if (HIST)
            a = __builtin_bit_cast(bf16x8, make_uint4(xin[k0 / 16][0], xin[k0 / 16][1], xin[k0 / 16][2],
                                                      xin[k0 / 16][3]));
        else
            a = rowValid ? LoadRow8(xr + k0 + kq) : zero8;
        bf16x8 b[MH / 32];
#pragma unroll
        for (int j = 0; j < MH / 32; ++j) b[j] = LoadRow8(&ws[buf][(j * 32 + r) * 16 + kq]);
#pragma unroll
        for (int j = 0; j < MH / 32; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], a, acc[j], 0, 0, 0);
        if (k0 + 16 < MI) slabStore(buf ^ 1, next);
        next = next2;
        __syncthreads();
    }
    hiddenOut(acc, OFF_B1);
    __syncthreads();

    // ---- layer 2: [32 x MH] x [MH x MH]
#pragma unroll
    for (int j = 0; j < MH / 32; ++j) acc[j] = f32x16{};
    // Layer 1's last barrier has passed: every wave is done with both slab buffers.
    next = slabLoad(OFF_W2, MH, 16);
    slabStore(0, slabLoad(OFF_W2, MH, 0));
    __syncthreads();
#pragma unroll
    for (int k0 = 0; k0 < MH; k0 += 16) {
        const int buf = (k0 / 16) & 1;
        uint4 next2{};
        if (k0 + 32 < MH) next2 = slabLoad(OFF_W2, MH, k0 + 32);
        const bf16x8 a = LoadRow8(hp(r, k0 + kq));
        bf16x8 b[MH / 32];
#pragma unroll
        for (int j = 0; j < MH / 32; ++j) b[j] = LoadRow8(&ws[buf][(j * 32 + r) * 16 + kq]);
#pragma unroll
        for (int j = 0; j < MH / 32; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], a, acc[j], 0, 0, 0);
        if (k0 + 16 < MH) slabStore(buf ^ 1, next);
        next = next2;
        __syncthreads();
    }
    hiddenOut(acc, OFF_B2);
    __syncthreads();

    // ---- layer 3: [32 x MH] x [MH x MO], one 32-column tile of which MO columns are real
    f32x16 out = f32x16{};
    bf16x8 b3[MH / 16];   // all of this lane's layer-3 weights in flight at once
#pragma unroll
    for (int k = 0; k < MH / 16; ++k) b3[k] = r < MO ? LoadRow8(Wb + OFF_W3 + (size_t)r * MH + 16 * k + kq) : zero8;
#pragma unroll
    for (int k = 0; k < MH / 16; ++k) {
        const bf16x8 a = LoadRow8(hp(r, 16 * k + kq));
        out = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b3[k], a, out, 0, 0, 0);
    }
    if (rowValid) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int f = outRow(i);
            if (f < MO) y[(m0 + r) * MO + f] = out[i] + P[OFF_B3 + f];
        }
    }
}

// Forward pass over `rows` inputs into y.
static int32_t Forward(const hwpa_initializer* m, const uint16_t* x, uint32_t rows, float* y, hipStream_t s)
{
    if (rows == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp forward: no rows");
    if (((uintptr_t)x & 15) != 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp forward: input not 16-byte aligned");
    const uint32_t per = (uint32_t)(kFusedRows * kFusedWaves);
    hipLaunchKernelGGL(MlpFusedForwardKernel<false>, dim3((rows + per - 1) / per), dim3(64 * kFusedWaves), 0, s, x,
                       nullptr, rows,
                       m->Pb, m->P, y);
    return CheckLaunch("MlpFusedForwardKernel");
}

// Inference straight from lane histograms: FeaturesKernel + Forward in one launch.
static int32_t ForwardFromHist(const hwpa_initializer* m, const hwpa_lane_hist* hist, uint32_t lanes, float* y,
                               hipStream_t s)
{
    if (lanes == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp forward: no lanes");
    // Whole lanes, so every wave's 32 rows are all valid or all past the end: the
    // HIST input staging reads a wave's half-lane of counters only when m0 < rows.
    static_assert(LS % kFusedRows == 0, "a wave's rows lie in one lane");
    const uint32_t rows = lanes * (uint32_t)LS;
    const uint32_t per = (uint32_t)(kFusedRows * kFusedWaves);
    hipLaunchKernelGGL(MlpFusedForwardKernel<true>, dim3((rows + per - 1) / per), dim3(64 * kFusedWaves), 0, s, nullptr,
                       hist, rows,
                       m->Pb, m->P, y);
    return CheckLaunch("MlpFusedForwardKernel");
}

// Mean loss of a batch into m->lossDev; its gradients into m->G, or (step given) applied.
static int32_t Backward(hwpa_initializer* m, const uint16_t* x, const float* t, const uint8_t* valid, uint32_t batch,
                        const AdamArgs* step, hipStream_t s)
{
    const uint32_t blocks = (uint32_t)(((uint64_t)batch + kTrainRows - 1) / kTrainRows);
    hipLaunchKernelGGL(TrainRowsKernel, dim3(blocks), dim3(64 * kTrainWaves), 0, s, x, t,
                       valid, batch, m->Pb, m->WT, m->P, m->omap, m->acts);
    int32_t rc = CheckLaunch("TrainRowsKernel");
    if (rc != HWPA_OK) return rc;
    const dim3 grid(kGradTiles + 1), threads(64 * kGradWaves);
    if (step)
        hipLaunchKernelGGL(TrainGradKernel<true>, grid, threads, 0, s, m->acts, batch, nullptr, m->lossDev, *step);
    else
        hipLaunchKernelGGL(TrainGradKernel<false>, grid, threads, 0, s, m->acts, batch, m->G, m->lossDev, AdamArgs{});
    return CheckLaunch("TrainGradKernel");
}

// Deterministic He-uniform initialisation from a 64-bit seed (biases zero).
static void InitParams(std::vector<float>& p, uint64_t seed)
{
    p.assign(NPARAM, 0.0f);
    uint64_t state = seed ^ 0x6a09e667f3bcc909ull;
    auto next = [&]() {
        state += 0x9e3779b97f4a7c15ull;
        uint64_t z = state;
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        z ^= z >> 31;
        return ((double)(z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](size_t off, int fanOut, int fanIn) {
        const double lim = std::sqrt(6.0 / fanIn);
        for (size_t i = 0; i < (size_t)fanOut * fanIn; ++i) p[off + i] = (float)((2.0 * next() - 1.0) * lim);
    };
    fill(OFF_W1, MH, MI);
    fill(OFF_W2, MH, MH);
    fill(OFF_W3, MO, MH);
}

int32_t MlpFeatures(const hwpa_lane_hist* hist, uint32_t lanes, uint16_t* x, hipStream_t s)
{
    hipLaunchKernelGGL(FeaturesKernel, dim3(lanes), dim3(LS), 0, s, hist, x);
    return CheckLaunch("FeaturesKernel");
}

const float* MlpOutputMap(const hwpa_initializer* m) { return m->omap; }

int32_t MlpTargets(const hwpa_lane_hist* hist, const float* diag, uint32_t lanes, float minConf, float* t,
                   uint8_t* valid, hipStream_t s)
{
    hipLaunchKernelGGL(TargetsKernel, dim3(lanes), dim3(LS), 0, s, hist, diag, minConf, t, valid);
    return CheckLaunch("TargetsKernel");
}

int32_t MlpForwardFromHist(const hwpa_initializer* m, const hwpa_lane_hist* hist, uint32_t lanes, float* y,
                           hipStream_t s)
{
    return ForwardFromHist(m, hist, lanes, y, s);
}

}  // namespace hwpa

extern "C" {

int32_t hwpa_initializer_create(uint64_t seed, hwpa_initializer** out)
{
    if (!out) return Fail(HWPA_ERR_INVALID_ARG, "null argument");
    *out = nullptr;
    hwpa_initializer* m = new (std::nothrow) hwpa_initializer();
    if (!m) return Fail(HWPA_ERR_OOM, "out of host memory");
    int32_t rc = DeviceAlloc((void**)&m->P, NPARAM * 4, "mlp parameters");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->Pb, NPARAM * 2 + 16, "mlp parameters");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->G, NPARAM * 4, "mlp gradients");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->Mo, NPARAM * 4, "mlp moments");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->Ve, NPARAM * 4, "mlp moments");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->lossDev, 16, "mlp loss");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->omap, 20 * sizeof(float), "mlp output map");
    if (rc == HWPA_OK) rc = DeviceAlloc((void**)&m->WT, NTRANS * 2, "mlp parameters");
    if (rc != HWPA_OK) {
        hwpa_initializer_destroy(m);
        return rc;
    }
    // Identity output map, unit weights, until the trainer sets one.
    for (int j = 0; j < 6; ++j) {
        m->omapHost[j] = 0.0f;
        m->omapHost[6 + j] = 1.0f;
        m->omapHost[12 + j] = 1.0f;
    }
    m->omapHost[18] = 1.0f;
    m->omapHost[19] = 1.0f;
    if (hipMemcpy(m->omap, m->omapHost, sizeof(m->omapHost), hipMemcpyHostToDevice) != hipSuccess) {
        hwpa_initializer_destroy(m);
        return Fail(HWPA_ERR_HIP, "output map upload failed");
    }
    std::vector<float> p;
    InitParams(p, seed);
    if ((rc = hwpa_initializer_set_params(m, p.data(), p.size())) != HWPA_OK) {
        hwpa_initializer_destroy(m);
        return rc;
    }
    *out = m;
    return HWPA_OK;
}

int32_t hwpa_initializer_destroy(hwpa_initializer* m)
{
    if (!m) return HWPA_OK;
    (void)hipDeviceSynchronize();
    FreeTrain(m);
    DeviceFree(m->P);
    DeviceFree(m->Pb);
    DeviceFree(m->G);
    DeviceFree(m->Mo);
    DeviceFree(m->Ve);
    DeviceFree(m->lossDev);
    DeviceFree(m->omap);
    DeviceFree(m->WT);
    LearnedWsFree(m->ws);
    delete m;
    return HWPA_OK;
}

int32_t hwpa_initializer_get_params(const hwpa_initializer* m, float* host_params, size_t n)
{
    if (!m || !host_params) return Fail(HWPA_ERR_INVALID_ARG, "null argument");
    if (n != NPARAM) return Fail(HWPA_ERR_INVALID_ARG, "parameter count must be HWPA_MLP_PARAMS");
    HWPA_HIP(hipDeviceSynchronize());
    HWPA_HIP(hipMemcpy(host_params, m->P, NPARAM * 4, hipMemcpyDeviceToHost));
    return HWPA_OK;
}

int32_t hwpa_initializer_set_params(hwpa_initializer* m, const float* host_params, size_t n)
{
    if (!m || !host_params) return Fail(HWPA_ERR_INVALID_ARG, "null argument");
    if (n != NPARAM) return Fail(HWPA_ERR_INVALID_ARG, "parameter count must be HWPA_MLP_PARAMS");
    HWPA_HIP(hipDeviceSynchronize());
    HWPA_HIP(hipMemcpy(m->P, host_params, NPARAM * 4, hipMemcpyHostToDevice));
    HWPA_HIP(hipMemset(m->Mo, 0, NPARAM * 4));
    HWPA_HIP(hipMemset(m->Ve, 0, NPARAM * 4));
    HWPA_HIP(hipMemset(m->G, 0, NPARAM * 4));
    m->step = 0;
    hipLaunchKernelGGL(ToBf16Kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, nullptr, m->P, m->Pb, m->WT,
                       (uint32_t)NPARAM);
    int32_t rc = CheckLaunch("ToBf16Kernel");
    if (rc != HWPA_OK) return rc;
    HWPA_HIP(hipDeviceSynchronize());
    return HWPA_OK;
}

int32_t hwpa_initializer_set_output_map(hwpa_initializer* m, const float offset[6], const float scale[6],
                                        const float weight[7])
{
    if (!m || !offset || !scale || !weight) return Fail(HWPA_ERR_INVALID_ARG, "null argument");
    for (int j = 0; j < 6; ++j) {
        if (!(scale[j] > 0.0f) || !hw_isfinite(offset[j]) || !(weight[j] >= 0.0f))
            return Fail(HWPA_ERR_INVALID_ARG, "output map: scales must be positive, weights non-negative");
    }
    if (!(weight[6] >= 0.0f) || !(weight[7] >= 0.0f))
        return Fail(HWPA_ERR_INVALID_ARG, "output map: weights must be non-negative");
    for (int j = 0; j < 6; ++j) {
        m->omapHost[j] = offset[j];
        m->omapHost[6 + j] = scale[j];
        m->omapHost[12 + j] = weight[j];
    }
    m->omapHost[18] = weight[6];
    m->omapHost[19] = weight[7];
    HWPA_HIP(hipDeviceSynchronize());
    HWPA_HIP(hipMemcpy(m->omap, m->omapHost, sizeof(m->omapHost), hipMemcpyHostToDevice));
    return HWPA_OK;
}

int32_t hwpa_initializer_get_output_map(const hwpa_initializer* m, float out[20])
{
    if (!m || !out) return Fail(HWPA_ERR_INVALID_ARG, "null argument");
    for (int j = 0; j < 20; ++j) out[j] = m->omapHost[j];
    return HWPA_OK;
}

int32_t hwpa_mlp_features(const hwpa_lane_hist* d_hist, uint32_t lanes, uint16_t* d_x, void* stream)
{
    if (!d_hist || !d_x || lanes == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp features: null argument or no lanes");
    if (((uintptr_t)d_x & 15) != 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp features: output must be 16-byte aligned");
    return MlpFeatures(d_hist, lanes, d_x, (hipStream_t)stream);
}

int32_t hwpa_mlp_targets(const hwpa_lane_hist* d_hist, const float* d_diag, uint32_t lanes, float min_confidence,
                         float* d_t, uint8_t* d_valid, void* stream)
{
    if (!d_hist || !d_diag || !d_t || !d_valid || lanes == 0)
        return Fail(HWPA_ERR_INVALID_ARG, "mlp targets: null argument or no lanes");
    return MlpTargets(d_hist, d_diag, lanes, min_confidence, d_t, d_valid, (hipStream_t)stream);
}

int32_t hwpa_mlp_forward(hwpa_initializer* m, const uint16_t* d_x, uint32_t rows, float* d_y, void* stream)
{
    if (!m || !d_x || !d_y || rows == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp forward: null argument or no rows");
    if (((uintptr_t)d_x & 15) != 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp forward: input must be 16-byte aligned");
    return Forward(m, d_x, rows, d_y, (hipStream_t)stream);
}

int32_t hwpa_mlp_forward_hist(hwpa_initializer* m, const hwpa_lane_hist* d_hist, uint32_t lanes, float* d_y,
                              void* stream)
{
    if (!m || !d_hist || !d_y || lanes == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp forward: null argument or no lanes");
    return ForwardFromHist(m, d_hist, lanes, d_y, (hipStream_t)stream);
}

int32_t hwpa_mlp_gradients(hwpa_initializer* m, const uint16_t* d_x, const float* d_t, const uint8_t* d_valid,
                           uint32_t batch, float* d_grads, float* d_loss, void* stream)
{
    if (!m || !d_x || !d_t || batch == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp gradients: null argument or empty batch");
    if (((uintptr_t)d_x & 15) != 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp gradients: input must be 16-byte aligned");
    int32_t rc = EnsureBatch(m, batch);
    if (rc != HWPA_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    if ((rc = Backward(m, d_x, d_t, d_valid, batch, nullptr, s)) != HWPA_OK) return rc;
    if (d_grads) HWPA_HIP(hipMemcpyAsync(d_grads, m->G, NPARAM * 4, hipMemcpyDeviceToDevice, s));
    if (d_loss) HWPA_HIP(hipMemcpyAsync(d_loss, m->lossDev, 4, hipMemcpyDeviceToDevice, s));
    return HWPA_OK;
}

int32_t hwpa_mlp_train_step(hwpa_initializer* m, const uint16_t* d_x, const float* d_t, const uint8_t* d_valid,
                            uint32_t batch, float lr, float* d_loss, void* stream)
{
    if (!m || !d_x || !d_t || batch == 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp train: null argument or empty batch");
    if (((uintptr_t)d_x & 15) != 0) return Fail(HWPA_ERR_INVALID_ARG, "mlp train: input must be 16-byte aligned");
    if (!(lr > 0.0f)) return Fail(HWPA_ERR_INVALID_ARG, "mlp train: learning rate must be positive");
    int32_t rc = EnsureBatch(m, batch);
    if (rc != HWPA_OK) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int64_t step = m->step + 1;
    const double b1 = 0.9, b2 = 0.999;
    const float c1 = (float)(1.0 - std::pow(b1, (double)step));
    const float c2 = (float)(1.0 - std::pow(b2, (double)step));
    const AdamArgs adam{m->P, m->Mo, m->Ve, m->Pb, m->WT, lr, (float)b1, (float)b2, c1, c2, 1e-8f};
    if ((rc = Backward(m, d_x, d_t, d_valid, batch, &adam, s)) != HWPA_OK) return rc;
    m->step = step;
    if (d_loss) HWPA_HIP(hipMemcpyAsync(d_loss, m->lossDev, 4, hipMemcpyDeviceToDevice, s));
    return HWPA_OK;
}

}  // extern "C"
