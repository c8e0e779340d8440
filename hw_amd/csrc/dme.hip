// dme.hip -- detection-model estimation: model initialisation from baseline
// statistics and the grouped-data EM fit of the 5-component mixture
// (DmeEmHost, traceAnalysis/DmeEmHost.cpp:131-925; DetectionModelHost
// update/export, traceAnalysis/DetectionModelHost.cpp:69-285).
//
// Mapping: one wave64 per lane, one thread per ZMW.  The only coupling
// between ZMWs is the EM early exit, which the reference takes when every ZMW
// of the lane has converged or failed (DmeEmHost.cpp:485); here that is one
// wave vote per iteration.  Each EM iteration is one pass over the 301 bin
// boundaries in registers: the M-step's baseline-variance sum is carried in
// the same pass (no per-boundary scratch).  All arithmetic keeps the CPU
// restatement's operation order so results match it bit for bit.

#include "internal.h"

#include <algorithm>
#include <cfloat>
#include <mutex>

namespace hwpa {

struct DmeDevCfg {
    float blVarMin, blVarMax, blVarNominal, signalScaler, shotVarCoeff;
    float refSnr;
    float relAmp[NA], cv[NA];
    float mixThresh0, mixThresh1, scaleSnrConfTol, pulseAmpReg, snrDrop, snrThresh0, snrThresh1, successThresh;
    float hl0, hl1;
    float log2pi;
    int32_t iterLimit;
    int32_t iterToLimit;
    int32_t updateMethod;
};

static DmeDevCfg MakeDevCfg(const hwpa_config& c)
{
    DmeDevCfg d{};
    const DmeConsts k = MakeDmeConsts(c);
    d.blVarMin = k.blVarMin;
    d.blVarMax = k.blVarMax;
    d.blVarNominal = k.blVarNominal;
    d.signalScaler = k.signalScaler;
    d.shotVarCoeff = k.shotVarCoeff;
    d.refSnr = c.movie.ref_snr;
    for (int a = 0; a < NA; ++a) {
        d.relAmp[a] = c.movie.analogs[a].rel_amplitude;
        d.cv[a] = c.movie.analogs[a].excess_noise_cv;
    }
    d.mixThresh0 = c.analog_mix_fraction_threshold[0];
    d.mixThresh1 = c.analog_mix_fraction_threshold[1];
    d.scaleSnrConfTol = c.scale_snr_conf_tol;
    d.pulseAmpReg = c.pulse_amp_regularization;
    d.snrDrop = c.snr_drop_thresh;
    d.snrThresh0 = c.min_analog_snr_thresh0;
    d.snrThresh1 = c.min_analog_snr_thresh1;
    d.successThresh = c.success_confidence_thresh;
    d.hl0 = c.confidence_half_life[0];
    d.hl1 = c.confidence_half_life[1];
    d.log2pi = std::log(2.0f * 3.1415926536f);   // libm, scalar (DmeEmHost.cpp:380)
    d.iterLimit = (int32_t)c.em_iteration_limit;
    d.iterToLimit = c.iterate_to_limit;
    d.updateMethod = (int32_t)c.model_update_method;
    return d;
}

struct Mode {
    float w, mean, var;
};
struct Model {
    Mode bl;
    Mode an[NA];
    float conf;
};

__device__ __forceinline__ float Covar(const DmeDevCfg& d, float cv2, float mean, float blVar)
{
    float r = blVar;
    r += d.shotVarCoeff * mean;
    r += cv2 * (mean * mean);
    return r;
}

__device__ __forceinline__ float Variance(float m0, float m1, float m2)
{
    float var = m1 * m1 / m0;
    var = (m2 - var) / (m0 - 1.0f);
    var = hw_maxf(var, 0.0f);
    return (m0 > 1.0f) ? var : hw_u2f(0x7fc00000u);
}

__device__ Model LoadModel(const hwpa_lane_model& m, int z)
{
    Model r;
    r.bl.w = hw_h2f(m.baseline.weights[z]);
    r.bl.mean = hw_h2f(m.baseline.means[z]);
    r.bl.var = hw_h2f(m.baseline.vars[z]);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        r.an[a].w = hw_h2f(m.analogs[a].weights[z]);
        r.an[a].mean = hw_h2f(m.analogs[a].means[z]);
        r.an[a].var = hw_h2f(m.analogs[a].vars[z]);
    }
    r.conf = hw_h2f(m.confidence[z]);
    return r;
}

__device__ void StoreModel(const Model& r, hwpa_lane_model& m, int z)
{
    m.baseline.weights[z] = hw_f2h(r.bl.w);
    m.baseline.means[z] = hw_f2h(r.bl.mean);
    m.baseline.vars[z] = hw_f2h(hw_minf(r.bl.var, 65000.0f));
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        m.analogs[a].weights[z] = hw_f2h(r.an[a].w);
        m.analogs[a].means[z] = hw_f2h(r.an[a].mean);
        m.analogs[a].vars[z] = hw_f2h(hw_minf(r.an[a].var, 65000.0f));
    }
    m.confidence[z] = hw_f2h(r.conf);
}

// DetectionModelHost::Update0/1/2 + Update(other) (DetectionModelHost.cpp:69-205)
__device__ void UpdateConf(const DmeDevCfg& d, Model& t, const Model& o)
{
    const float confSum = t.conf + o.conf;
    const float f = (confSum > 0.0f) ? o.conf / confSum : 0.0f;
    const float a = 1.0f - f;
    const float b = f;
    if (d.updateMethod == 0) {
        t.bl.mean = a * t.bl.mean + b * o.bl.mean;
        t.bl.var = a * t.bl.var + b * o.bl.var;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            t.an[i].mean = a * t.an[i].mean + b * o.an[i].mean;
            t.an[i].var = a * t.an[i].var + b * o.an[i].var;
        }
    } else {
        const float prevBlVar = t.bl.var;
        const float bw = a * t.bl.w + b * o.bl.w;
        t.bl.w = bw;
        t.bl.mean = a * t.bl.mean + b * o.bl.mean;
        const float bv = hw_dpowf(t.bl.var, a) * hw_dpowf(o.bl.var, b);
        t.bl.var = bv;
        const float aw = 0.25f * (1.0f - bw);
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            t.an[i].w = aw;
            float cv2;
            if (d.updateMethod == 2) {
                float tx = t.an[i].var - prevBlVar;
                tx -= t.an[i].mean * d.shotVarCoeff;
                tx /= (t.an[i].mean * t.an[i].mean);
                float ox = o.an[i].var - o.bl.var;
                ox -= o.an[i].mean * d.shotVarCoeff;
                ox /= (o.an[i].mean * o.an[i].mean);
                cv2 = a * tx + b * ox;
            } else {
                cv2 = d.cv[i] * d.cv[i];
            }
            const float am = hw_dpowf(t.an[i].mean, a) * hw_dpowf(o.an[i].mean, b);
            t.an[i].mean = am;
            t.an[i].var = Covar(d, cv2, am, bv);
        }
    }
    t.conf = confSum;
}

// DmeEmHost::InitLaneDetModel (DmeEmHost.cpp:871-925)
__global__ __launch_bounds__(64) void DmeInitKernel(const hwpa_baseliner_stats* stats, hwpa_lane_model* models,
                                                    DmeDevCfg d)
{
    const hwpa_baseliner_stats& s = stats[blockIdx.x];
    hwpa_lane_model& m = models[blockIdx.x];
    const int z = threadIdx.x;
    const float m0 = s.baseline.m0[z], m1 = s.baseline.m1[z], m2 = s.baseline.m2[z];
    const float blWeight = m0 / s.full.basic.m0[z];
    float blMean = m1 / m0 + s.baseline.offset[z];
    float blVar = Variance(m0, m1, m2);
    if (hw_isnan(blMean)) blMean = 0.0f;
    if (hw_isnan(blVar)) blVar = 100.0f;
    blVar = hw_clampf(blVar, d.blVarMin, d.blVarMax);
    m.confidence[z] = hw_f2h(0.1f);
    m.baseline.weights[z] = hw_f2h(blWeight);
    m.baseline.means[z] = hw_f2h(blMean);
    m.baseline.vars[z] = hw_f2h(blVar);
    const float amw = (1.0f - blWeight) / (float)NA;
    const float refSignal = d.refSnr * hw_sqrtf(blVar);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        m.analogs[a].weights[z] = hw_f2h(amw);
        const float aMean = hw_maxf(0.0f, blMean + d.relAmp[a] * refSignal);
        m.analogs[a].means[z] = hw_f2h(aMean);
        m.analogs[a].vars[z] = hw_f2h(Covar(d, d.cv[a] * d.cv[a], aMean, blVar));
    }
}

// Histogram view of one ZMW (UHistogramSimd(const LaneHistogram&), UHistogramSimd.cpp:100-118).
struct HistView {
    const hwpa_lane_hist* h;
    int z;
    float lb, bs;
    __device__ float Start(int b) const { return lb + (float)b * bs; }
    // Index NB is the always-empty overflow bin of UHistogramSimd (UHistogramSimd.cpp:66).
    __device__ uint32_t Cnt(int b) const { return (b < NB) ? (uint32_t)h->bin_count[b][z] : 0u; }
};

// Bins read at once by the set-up passes over a ZMW's counts: the loads of a batch are
// all in flight together (a loop that tests each count before it loads the next waits for
// memory at every bin: 90 of the 1070 us that one wave's estimate took).
constexpr int kSetupBatch = 20;
static_assert(NB % kSetupBatch == 0, "whole set-up batches");

// Total of the in-range counts (16-bit, as UHistogramSimd adds them), the last nonempty bin
// and the counts' sum as the EM's float accumulation gives it.
__device__ uint32_t InRange(const HistView& h, int* lastNonzero, float* floatSum)
{
    uint32_t s = 0;
    int last = -1;
#pragma unroll 1
    for (int b = 0; b < NB; b += kSetupBatch) {
        uint32_t c[kSetupBatch];
#pragma unroll
        for (int j = 0; j < kSetupBatch; ++j) c[j] = h.Cnt(b + j);
#pragma unroll
        for (int j = 0; j < kSetupBatch; ++j) {
            s += c[j];
            last = c[j] ? b + j : last;
        }
    }
    *lastNonzero = last;
    // Every partial sum below 2^24 is exact in float, so the order does not matter there.
    float f = (float)s;
    if (s >= (1u << 24)) {
        f = 0.0f;
        for (int b = 0; b < NB; ++b) f += (float)h.Cnt(b);
    }
    *floatSum = f;
    return s & 0xffffu;
}

// UHistogramSimd::CumulativeCount (UHistogramSimd.cpp:199-238)
__device__ float CumulativeCount(const HistView& h, uint32_t lowOut, uint32_t inRange, float x)
{
    const bool mNan = hw_isnan(x);
    const bool mLow = x < h.Start(0);
    const bool mHigh = x >= h.Start(NB);
    const bool mIn = !(mNan || mLow || mHigh);
    int xbin = hw_floor_i32((x - h.Start(0)) / h.bs);
    if (!mIn || xbin < 0) xbin = 0;   // (x inside NaN bounds: the quotient is NaN, and so is the result)
    const float xrem = x - h.Start(xbin);
    const float xbinCount = (float)h.Cnt(xbin);
    float cc = (float)lowOut;
    uint32_t below = 0;
#pragma unroll 1
    for (int b = 0; b < NB && __any(b < xbin); b += kSetupBatch) {
        uint32_t c[kSetupBatch];
#pragma unroll
        for (int j = 0; j < kSetupBatch; ++j) c[j] = h.Cnt(b + j);
#pragma unroll
        for (int j = 0; j < kSetupBatch; ++j) below += (b + j < xbin) ? c[j] : 0u;
    }
    cc += (float)(below & 0xffffu);
    cc += xbinCount * xrem / h.bs;
    if (mLow) cc = (float)lowOut;
    if (mHigh) cc = (float)((lowOut + inRange) & 0xffffu);
    if (mNan) cc = hw_u2f(0x7fc00000u);
    return cc;
}

// UHistogramSimd::Fractile (UHistogramSimd.cpp:140-197)
__device__ float Fractile(const HistView& h, uint32_t lowOut, uint32_t total, float frac)
{
    const float nfz = frac * (float)total;
    uint32_t n = lowOut;
    if (n > 0 && (float)n >= nfz) return hw_u2f(0xff800000u);
    // The first bin at which the running count (mod 2^16) is positive and reaches nfz.
    int i = 0;
    uint32_t niz = 0;
    bool go = n == 0 || (float)n < nfz;
#pragma unroll 1
    for (int b = 0; b < NB && __any(go); b += kSetupBatch) {
        uint32_t c[kSetupBatch];
#pragma unroll
        for (int j = 0; j < kSetupBatch; ++j) c[j] = h.Cnt(b + j);
#pragma unroll
        for (int j = 0; j < kSetupBatch; ++j) {
            if (go) {
                n = (n + c[j]) & 0xffffu;
                niz = c[j];
                ++i;
                go = n == 0 || (float)n < nfz;
            }
        }
    }
    if ((float)n < nfz) return hw_u2f(0x7f800000u);
    i -= 1;   // -1 (no bin taken) only for a NaN fraction, whose result is NaN
    const float x0 = h.Start(i);
    const int m = (int)n - (int)niz;
    return x0 + h.bs * (nfz - (float)m) / (float)(niz + 1);
}

__device__ __forceinline__ float Sum5Tree(const float* v) { return (v[0] + v[1]) + (v[2] + (v[3] + v[4])); }

enum { EM_PLAIN = 0, EM_LEARNED = 1 };

// Extra inputs/outputs of the EM kernel beyond the reference's.
struct EmExtra {
    const float* init;        // EM_LEARNED: network outputs [lane*64 + z][HWPA_MLP_OUT]
    const float* omap;        // EM_LEARNED: output map {off[6], scale[6], ...}
    uint8_t* fallback;        // EM_LEARNED: 1 = start rejected, model left for the plain EM
    float* diag;              // optional raw estimate [lane][HWPA_EM_DIAG_ROWS][64]
    const uint32_t* active;   // optional: number of valid ZMWs; lanes at or beyond it exit, and the
                              // last lane's missing ZMWs run as copies of its first one
    uint32_t activeMin, activeMax;   // with active: the launch does nothing unless activeMin <= *active <= activeMax
    const uint8_t* laneSel;   // optional: only lanes whose 64 flags here are all set run
    float acceptConf;         // EM_LEARNED: minimum confidence to accept the capped EM
    float convTol;            // EM_LEARNED: relative log-likelihood convergence tolerance
    int32_t iterLimit;        // EM_LEARNED: iteration cap
    float gateLogit;          // EM_LEARNED: network confidence logit below which the capped EM is skipped
    int32_t laneMinConf;      // EM_LEARNED: a lane with fewer ZMWs above the gate gates all of them
};

// DmeEmHost::EstimateLaneDetModel (DmeEmHost.cpp:216-615).  EM_LEARNED replaces
// the start model of the EM loop (after PrelimEstimate and the scale factor,
// which still set the amplitude prior) by the network's prediction, caps the
// iterations, uses its own log-likelihood convergence tolerance and accepts
// the result only for converged ZMWs with status OK and enough confidence.
// exp(t) rounds to +0 for every t below this (exp(-103.98) is 2^-150).
constexpr float kExpZeroBelow = -105.0f;
// Boundaries per exact restart of the density recurrence of the E-step.
constexpr int kRecurBlock = 10;
// hw_expf without its clamp and its NaN case, for finite t in [-8e6, 200] (and any t whose
// result is not used): the same steps, so the same bits.  Below -200 the clamp only keeps k in
// range: t log2(e) is within 0.7 of its rounded value there, so |r| < 0.9, exp(r)'s polynomial is
// positive and 2^k times it is +0, as with the clamp.
__device__ __forceinline__ float ExpBounded(float t)
{
    const float kf = hw_rintf(t * 1.44269502162933349609375f);
    const float r = hw_fmaf(-kf, 1.428606765330187045e-06f, hw_fmaf(-kf, 0.693145751953125f, t));
    return hw_ldexpf(hw_exp_poly(r), (int)kf);
}

// The E-step of small pools (QUAD): four threads per ZMW, a workgroup of four waves per lane, for
// launches that leave SIMDs without a wave.  The boundaries are taken in groups of four blocks:
// thread u forms block u's densities, bin probabilities, logs and weights, leaves them in LDS in
// boundary order, and then carries a quarter of the fourteen running sums over the group's 40
// boundaries: its analog's two, one of the baseline's four, and the probability's or the
// log-likelihood's.  Each sum is formed in the same order from the same terms, so the bits stay.
// What counts is the instructions of one wave, which issues one in four cycles: 131 thousand
// against 314 (and 14 thousand LDS accesses).  48 lanes in a running pool: 0.60 against 0.97 ms;
// start-up estimate: 48 lanes 0.74 against 1.27 ms, 256 lanes 0.75 against 1.33, 384 lanes (two
// rounds) 1.38 against 1.37.
constexpr int kQuadGroup = 4 * kRecurBlock;
constexpr int kQuadRow = kQuadGroup + 4;   // a row holds the boundary before the group too; 16-byte rows
enum { QR_D = 0, QR_F = 5, QR_G, QR_DEV, QR_W, QR_WD, QR_P, QR_N, QR_LG, QR_ROWS };
constexpr int kQuadZmw = QR_ROWS * kQuadRow;

// Value of quad thread P, and of the thread before in the quad (thread 0 gets thread 3's).
template <int P>
__device__ __forceinline__ float EmQuadAt(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), P * 0x55, 0xf, 0xf, true));
}
__device__ __forceinline__ float EmQuadPrev(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x93, 0xf, 0xf, true));   // [3, 0, 1, 2]
}

// MINW: waves per SIMD the registers allow (EmWavesPerSimd).  QUAD: see above.
template <int MODE, int MINW, bool QUAD = false>
__global__ __launch_bounds__(QUAD ? 4 * LS : LS, MINW) void DmeEstimateKernel(const hwpa_lane_hist* __restrict__ hists,
                                                        const hwpa_baseliner_stats* __restrict__ stats,
                                                        hwpa_lane_model* models, int32_t* iters, DmeDevCfg d,
                                                        float evolve, EmExtra x)
{
    const int lane = blockIdx.x;
    const int z = QUAD ? threadIdx.x >> 2 : threadIdx.x;
    const int u = QUAD ? threadIdx.x & 3 : 0;   // place in the quad; place 0 writes the results
    // Votes over the lane's 64 ZMWs.
    auto laneAll = [](bool v) -> bool { return QUAD ? __syncthreads_and(v ? 1 : 0) != 0 : (bool)__all(v); };
    auto laneCount = [&](bool v) -> int {
        return QUAD ? __syncthreads_count(v && u == 0 ? 1 : 0) : (int)__popcll(__ballot(v));
    };
    int zin = z;   // the ZMW whose inputs this thread reads
    if (x.active) {
        const uint32_t valid = *x.active;
        if (valid < x.activeMin || valid > x.activeMax) return;
        if ((uint32_t)lane * LS >= valid) return;
        if ((uint32_t)lane * LS + (uint32_t)z >= valid) zin = 0;
    }
    if (x.laneSel && !laneAll(x.laneSel[(size_t)lane * LS + z] != 0)) return;
    bool gated = false;       // EM_LEARNED: the network's confidence sends this ZMW to the plain EM
    if (MODE == EM_LEARNED) {
        // Confidence gate: a ZMW below it takes no capped iteration of its own (it still
        // runs in step with its lane, but counts as done and is rejected); a lane with fewer
        // than laneMinConf ZMWs above it sends all of them to the plain EM (its iterations
        // would cost the whole lane for those few).  A lane gated whole leaves its models
        // as they are, as every rejected ZMW does, and stops here.
        gated = !(x.init[((size_t)lane * LS + z) * HWPA_MLP_OUT + 11] >= x.gateLogit);
        if ((uint32_t)laneCount(!gated) < (uint32_t)x.laneMinConf) gated = true;
        if (laneAll(gated)) {
            x.fallback[(size_t)lane * LS + z] = 1;
            if (threadIdx.x == 0 && iters) iters[lane] = 0;
            return;
        }
    }
    // Tables of the E-step's log / reciprocal of bin probabilities, one entry per thread.
    __shared__ float sRc[HW_LOGTAB_N], sLc[HW_LOGTAB_N];
    static_assert(HW_LOGTAB_N == LS, "one table entry per thread");
    if (threadIdx.x < LS) hw_logtab_entry(threadIdx.x, &sRc[threadIdx.x], &sLc[threadIdx.x]);
    __shared__ __align__(16) float sQuad[QUAD ? LS * kQuadZmw : 1];
    __shared__ __align__(16) float sOnes[QUAD ? kQuadRow : 1];
    if (QUAD && threadIdx.x < (unsigned)kQuadRow) sOnes[threadIdx.x] = 1.0f;
    __syncthreads();
    const hwpa_lane_hist& lh = hists[lane];
    const hwpa_baseliner_stats& bs = stats[lane];
    hwpa_lane_model& lm = models[lane];

    HistView h{&lh, zin, lh.low_bound[zin], lh.bin_size[zin]};
    const uint32_t lowOut = lh.outlier_low[zin], highOut = lh.outlier_high[zin];
    int lastNz;
    float njSum;
    const uint32_t inRange = InRange(h, &lastNz, &njSum);
    const uint32_t numFrames = (inRange + ((lowOut + highOut) & 0xffffu)) & 0xffffu;

    const float rpa[NA] = {d.relAmp[0], d.relAmp[1], d.relAmp[2], d.relAmp[3]};
    const float rpaSqSum = (rpa[0] * rpa[0] + rpa[2] * rpa[2]) + (rpa[1] * rpa[1] + rpa[3] * rpa[3]);
    const float rpaMin = hw_minf(hw_minf(rpa[0], rpa[1]), hw_minf(rpa[2], rpa[3]));

    Model det = LoadModel(lm, zin);
    // A missing ZMW reads the model of the lane's first, which another wave writes at its end.
    if (QUAD && x.active) __syncthreads();
    det.conf *= evolve;

    // PrelimEstimate (DmeEmHost.cpp:161-214)
    {
        Model w = det;
        const float nBl = bs.baseline.m0[zin];
        const float total = bs.full.basic.m0[zin];
        const float blWeight = hw_maxf(nBl / total, 0.01f);
        const bool mask = nBl >= 3.0f;
        float blVar = mask ? Variance(bs.baseline.m0[zin], bs.baseline.m1[zin], bs.baseline.m2[zin]) : w.bl.var;
        blVar = hw_clampf(blVar, d.blVarMin, d.blVarMax);
        const float blMean = mask ? (bs.baseline.m1[zin] / bs.baseline.m0[zin] + bs.baseline.offset[zin]) : w.bl.mean;
        const float scale = hw_sqrtf(blVar / w.bl.var);
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const float mean = w.an[a].mean * scale;
            const float var = Covar(d, d.cv[a] * d.cv[a], mean, blVar);
            w.an[a].mean = mean;
            w.an[a].var = var;
            w.an[a].w = 0.25f * (1.0f - blWeight);
        }
        w.bl.w = blWeight;
        w.bl.mean = blMean;
        w.bl.var = blVar;
        float conf = 0.1f * hw_satlin(0.0f, 500.0f, nBl - 3.0f);
        conf *= hw_satlin(d.blVarMax, 0.5f * (d.blVarNominal + d.blVarMax), blVar);
        w.conf = conf;
        UpdateConf(d, det, w);
    }
    Model work = det;

    // PrelimScaleFactor (DmeEmHost.cpp:618-654) and ScaleModelSnr (:837-852)
    float scaleFactor;
    {
        const float bgSigma = hw_sqrtf(work.bl.var);
        const float thresh = 2.5f * bgSigma + work.bl.mean;
        const float bgCount = CumulativeCount(h, lowOut, inRange, thresh);
        const float totalCount = (float)((lowOut + inRange) & 0xffffu);
        const float fractile = 0.5f * (bgCount + totalCount) / totalCount;
        float avg = 0.0f;
#pragma unroll
        for (int a = 0; a < NA; ++a) avg += work.an[a].mean;
        avg /= (float)NA;
        const float w = hw_satlin(0.0f, d.scaleSnrConfTol, work.conf);
        float sf = Fractile(h, lowOut, numFrames, fractile) / avg;
        sf = (1.0f - w) * sf + w;
        scaleFactor = hw_minf(hw_maxf(sf, 0.1f), 10.0f);
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        work.an[a].mean = scaleFactor * work.an[a].mean;
        work.an[a].var = Covar(d, d.cv[a] * d.cv[a], work.an[a].mean, work.bl.var);
    }

    float rho[5], mu[5], var[5], rhoEst[5], muEst[5], varEst[5];
    const float rhoMin = 0.001f;
    rho[0] = hw_maxf(work.bl.w, rhoMin);
    mu[0] = work.bl.mean;
    var[0] = work.bl.var;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        rho[a + 1] = hw_maxf(work.an[a].w, rhoMin);
        mu[a + 1] = work.an[a].mean;
        var[a + 1] = work.an[a].var;
    }
    const float varQuant = (h.bs * h.bs) / 12.0f;
#pragma unroll
    for (int k = 0; k < 5; ++k) var[k] += varQuant;
    var[0] = hw_minf(var[0], d.blVarMax);
    {
        const float rs = Sum5Tree(rho);
#pragma unroll
        for (int k = 0; k < 5; ++k) rho[k] = rho[k] / rs;
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        rhoEst[k] = rho[k];
        muEst[k] = mu[k];
        varEst[k] = var[k];
    }
    float s = ((mu[1] * rpa[0] + mu[2] * rpa[1]) + (mu[3] * rpa[2] + mu[4] * rpa[3])) / rpaSqSum;
    const float sExpect = s / scaleFactor;
    const float sExpectWeight = det.conf * d.pulseAmpReg;
    float logLike = -FLT_MAX;
    const float binProbMin = hw_maxf((float)numFrames * h.bs, 1.0f) * FLT_MIN;
    int status = (numFrames < 160u) ? HWPA_ZS_INSUF_DATA : HWPA_ZS_OK;
    bool converged = false;
    float mlLogLike = hw_u2f(0xff800000u);
    const float halfBin = 0.5f * h.bs;
    int iterLimit = d.iterLimit;
    if (MODE == EM_LEARNED) {
        // Network start: output j < 6 stands for off[j] + scale[j] * y[j] in units
        // of u = 2 binSize from the lower bound (means) and log(var / u^2);
        // outputs 6..10 are softmax mixture logits.
        const float* y = x.init + ((size_t)lane * LS + z) * HWPA_MLP_OUT;
        const float u = 2.0f * h.bs;
        float r[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) r[j] = x.omap[j] + x.omap[6 + j] * y[j];
        float mx = y[6];
#pragma unroll
        for (int k = 1; k < 5; ++k) mx = hw_maxf(mx, y[6 + k]);
        float e[5], se = 0.0f;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            e[k] = hw_expf(y[6 + k] - mx);
            se += e[k];
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) rho[k] = hw_maxf(e[k] / se, rhoMin);
        const float rs = Sum5Tree(rho);
#pragma unroll
        for (int k = 0; k < 5; ++k) rho[k] = rho[k] / rs;
        mu[0] = h.lb + u * r[0];
        var[0] = hw_clampf((u * u) * hw_expf(r[1]), d.blVarMin, d.blVarMax);
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            mu[a + 1] = h.lb + u * r[2 + a];
            var[a + 1] = Covar(d, d.cv[a] * d.cv[a], mu[a + 1], var[0]);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            rhoEst[k] = rho[k];
            muEst[k] = mu[k];
            varEst[k] = var[k];
        }
        s = ((mu[1] * rpa[0] + mu[2] * rpa[1]) + (mu[3] * rpa[2] + mu[4] * rpa[3])) / rpaSqSum;
        iterLimit = x.iterLimit;
    }

    int it = 0;
    for (; it < iterLimit; ++it) {
        // ---- E-step
        float varinv[5], pref[5], nhv[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            varinv[k] = 1.0f / var[k];
            pref[k] = (hw_cephes_logf(rho[k]) - 0.5f * hw_cephes_logf(var[k])) - 0.5f * d.log2pi;
            nhv[k] = -0.5f * varinv[k];
        }
        // Every use of a responsibility is boundaryProb * tau_i = exp(t_i)
        // (DmeEmHost.cpp:431-432,547-548), so the boundary carries the component
        // densities dd_i = exp(t_i) and boundaryProb is their sum.  The bin sums of
        // the reference, sum_b (dd_i(b) + dd_i(b+1)) n_b / binProb_b, are taken per
        // boundary: sum_c dd_i(c) (f_{c-1} + f_c) with f_b = n_b / binProb_b, one fused
        // multiply-add per sum.  The baseline second moment of the M-step is
        // accumulated in the same pass about the pivot piv (this iteration's baseline
        // mean): q1 and q2 are the first and second moments of (x - piv) under the
        // baseline weights, shifted to the new mean after the M-step.  Waves skip
        // exact zeros: exps of boundaries where every t_i < -105 (exp rounds to +0),
        // and the sums of boundaries whose two bins are empty for all 64 ZMWs.
        const float piv = mu[0];
        float probSum = 0.0f, wps = 0.0f, q1 = 0.0f, q2 = 0.0f;
        float ci[5] = {0.f, 0.f, 0.f, 0.f, 0.f}, mom1[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        // Densities along the boundaries x_c = lb + c bs: t_i is quadratic in c, so
        // dd_i(c+1) = dd_i(c) R_i(c) with R_i(c) = exp(t_i(c+1) - t_i(c)) and
        // R_i(c+1) = R_i(c) Q_i, Q_i = exp(-bs^2 / var_i): two multiplies per density.
        // Every kRecurBlock boundaries dd_i and R_i are recomputed from exp.  The products
        // follow the ideal grid x_c + j bs; against exp at the rounded boundaries they
        // differ by |x - mu| / var times the boundary's rounding (below 1e-4 relative
        // within 14 sigma of the mean, 1e-5 near it).  A ZMW whose density at the
        // restart is below FLT_MIN while rising, or whose ratio exceeds e^80, takes exp
        // at every boundary of the block (a density coming out of underflow cannot be
        // continued from +0).
        float dd[5], rr[5], qq[5], nbs[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            qq[k] = hw_expf((2.0f * nhv[k]) * (h.bs * h.bs));
            nbs[k] = nhv[k] * h.bs;
        }
        auto tAt = [&](float x, int i) {
            const float y = x - mu[i];
            return hw_fmaf(y * y, nhv[i], pref[i]);
        };
        // Whether every exponent of this iteration's restarts lies in [-8e6, 200] for all ZMWs
        // of the wave: then ExpBounded serves them (not the case only for degenerate models or
        // bounds: NaN, infinite, zero or negative variances).
        // nanComp: this ZMW's components with a NaN parameter, whose density is NaN everywhere
        // (a product as well as an exp of NaN), so they never need an exp per boundary.
        bool bounded = true;
        uint32_t nanComp = 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            nanComp |= (hw_isnan(pref[i]) || hw_isnan(mu[i]) || hw_isnan(nhv[i]) ? 1u : 0u) << i;
            const float far = __builtin_fmaxf(hw_fabsf(h.lb - mu[i]), hw_fabsf(h.Start(NB) - mu[i]));
            bounded = bounded && nhv[i] <= 0.0f && (far * far) * nhv[i] >= -4e6f && pref[i] <= 80.0f && pref[i] >= -1e6f;
        }
        bounded = __all(bounded);
        float maxMu = mu[0];
#pragma unroll
        for (int k = 1; k < 5; ++k) maxMu = hw_maxf(maxMu, mu[k]);
        if constexpr (QUAD) {
            float* q = sQuad + z * kQuadZmw;
            auto row = [&](int r) -> float* { return q + r * kQuadRow; };
            // This thread's sums: own[c] += A B for its analog's two, the baseline's one and (0)
            // the probability's or (1) the log-likelihood's.
            float own = 0.0f, ownX = 0.0f, base = 0.0f, acc = 0.0f;
            const float* baseA = u < 2 ? row(QR_D) : u == 2 ? row(QR_W) : row(QR_WD);
            const float* baseB = u == 0 ? row(QR_F) : u == 1 ? row(QR_G) : row(QR_DEV);
            const float* accA = u == 0 ? row(QR_P) : row(QR_N);
            const float* accB = u == 0 ? sOnes : row(QR_LG);
            const float* ownD = row(QR_D + 1 + u);
            float bpC = 0.0f, fC = 0.0f, d0C = 0.0f;   // of the boundary before the group
            float fFirst = 0.0f;                       // weight of the bin before the thread's block
            row(QR_D + 1 + u)[0] = 0.0f;
            if (u == 0) row(QR_D)[0] = 0.0f;
            auto count = [&](int c) -> uint32_t {      // of the bin before boundary c
                return (uint32_t)lh.bin_count[min(max(c - 1, 0), NB - 1)][zin];
            };
            uint32_t cn[kRecurBlock];
#pragma unroll
            for (int j = 0; j < kRecurBlock; ++j) cn[j] = count(kRecurBlock * u + j);
            int cLast = NB, at = NB % kQuadGroup + 1;   // the last boundary taken, its place in the rows
#pragma unroll 1
            for (int g0 = 0; g0 <= NB; g0 += kQuadGroup) {
                if (g0 > 0) {
                    const float tol = hw_ldexpf(EmQuadAt<0>(acc), -27);
                    const bool tail = lastNz < g0 - 1 && h.Start(g0 - 1) > maxMu && h.bs * bpC < tol && binProbMin < tol;
                    if (__all(tail)) {
                        cLast = g0 - 1;
                        at = 0;
                        break;
                    }
                }
                const int c0 = g0 + kRecurBlock * u;   // the thread's first boundary
                uint32_t exMask = 0;
                {
                    const float x0 = h.Start(c0), x1 = h.Start(c0 + kRecurBlock);
#pragma unroll
                    for (int i = 0; i < 5; ++i) {
                        const float y0 = x0 - mu[i];
                        const float t0 = hw_fmaf(y0 * y0, nhv[i], pref[i]);
                        const float dl = nbs[i] * hw_fmaf(2.0f, y0, h.bs);
                        if (bounded) {
                            dd[i] = ExpBounded(t0);
                            rr[i] = ExpBounded(dl);
                        } else {
                            dd[i] = hw_expf(t0);
                            rr[i] = hw_expf(dl);
                        }
                        const bool rec = (dd[i] >= FLT_MIN || dl <= 0.0f) && dl <= 80.0f;
                        const bool flat = t0 < kExpZeroBelow && tAt(x1, i) < kExpZeroBelow && x1 <= mu[i];
                        if ((!rec && flat) || t0 < kExpZeroBelow) rr[i] = 0.0f;   // +0 from here on, or an exp below
                        exMask |= (!rec && !flat && ((nanComp >> i) & 1u) == 0u && c0 < NB ? 1u : 0u) << i;
                    }
                }
                const bool anyEx = __any(exMask != 0u);
                float bp[kRecurBlock], f[kRecurBlock], d0[kRecurBlock];
#pragma unroll
                for (int j = 0; j < kRecurBlock; ++j) {
                    if (j > 0) {
#pragma unroll
                        for (int i = 0; i < 5; ++i) {
                            dd[i] = dd[i] * rr[i];
                            rr[i] = rr[i] * qq[i];
                        }
                        if (anyEx) {
                            const float x = h.Start(c0 + j);
#pragma unroll
                            for (int i = 0; i < 5; ++i)
                                if ((exMask >> i) & 1u) dd[i] = hw_expf(tAt(x, i));
                        }
                    }
                    const bool in = c0 + j <= NB;
                    bp[j] = in ? Sum5Tree(dd) : 0.0f;
                    d0[j] = in ? dd[0] : 0.0f;
#pragma unroll
                    for (int i = 0; i < 5; ++i) row(QR_D + i)[kRecurBlock * u + j + 1] = in ? dd[i] : 0.0f;
                }
                const float bpB = EmQuadPrev(bp[kRecurBlock - 1]);
                float bpPrev = u == 0 ? bpC : bpB;
                bpC = EmQuadAt<3>(bp[kRecurBlock - 1]);
#pragma unroll
                for (int j = 0; j < kRecurBlock; ++j) {
                    const bool in = c0 + j <= NB && (j > 0 || c0 > 0);   // (no bin before boundary 0)
                    const float binp = hw_max_pos(halfBin * (bpPrev + bp[j]), binProbMin);
                    bpPrev = bp[j];
                    const float nj = in ? (float)cn[j] : 0.0f;
                    float lg, rcp;
                    hw_log_rcp_tab(binp, sRc, sLc, &lg, &rcp);
                    f[j] = nj * rcp;
                    const int p = kRecurBlock * u + j;
                    row(QR_P)[p] = in ? binp : 0.0f;
                    row(QR_N)[p] = nj;
                    row(QR_LG)[p] = lg;
                    cn[j] = count(c0 + kQuadGroup + j);
                }
                const float fB = EmQuadPrev(f[kRecurBlock - 1]), d0B = EmQuadPrev(d0[kRecurBlock - 1]);
                float fPrev = u == 0 ? fC : fB, d0Prev = u == 0 ? d0C : d0B;
                fC = EmQuadAt<3>(f[kRecurBlock - 1]);
                d0C = EmQuadAt<3>(d0[kRecurBlock - 1]);
                fFirst = f[0];
#pragma unroll
                for (int j = 0; j < kRecurBlock; ++j) {
                    // Terms of boundary c0 + j - 1.
                    const bool in = c0 + j <= NB;
                    const float x = h.Start(c0 + j - 1);
                    const float F = in ? fPrev + f[j] : 0.0f;
                    const float dev = x - piv;
                    const float w = d0Prev * F;
                    const int p = kRecurBlock * u + j;
                    row(QR_F)[p] = F;
                    row(QR_G)[p] = x * F;
                    row(QR_DEV)[p] = dev;
                    row(QR_W)[p] = w;
                    row(QR_WD)[p] = w * dev;
                    fPrev = f[j];
                    d0Prev = d0[j];
                }
                // The rows pass between lanes of one wave only; its LDS accesses stay in order.
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll 2
                for (int p = 0; p < kQuadGroup; p += 4) {
                    const float4 vd = *reinterpret_cast<const float4*>(ownD + p);
                    const float4 vF = *reinterpret_cast<const float4*>(row(QR_F) + p);
                    const float4 vG = *reinterpret_cast<const float4*>(row(QR_G) + p);
                    const float4 a = *reinterpret_cast<const float4*>(baseA + p);
                    const float4 b = *reinterpret_cast<const float4*>(baseB + p);
                    const float4 ea = *reinterpret_cast<const float4*>(accA + p);
                    const float4 eb = *reinterpret_cast<const float4*>(accB + p);
                    own = hw_fmaf(vd.x, vF.x, own);
                    own = hw_fmaf(vd.y, vF.y, own);
                    own = hw_fmaf(vd.z, vF.z, own);
                    own = hw_fmaf(vd.w, vF.w, own);
                    ownX = hw_fmaf(vd.x, vG.x, ownX);
                    ownX = hw_fmaf(vd.y, vG.y, ownX);
                    ownX = hw_fmaf(vd.z, vG.z, ownX);
                    ownX = hw_fmaf(vd.w, vG.w, ownX);
                    base = hw_fmaf(a.x, b.x, base);
                    base = hw_fmaf(a.y, b.y, base);
                    base = hw_fmaf(a.z, b.z, base);
                    base = hw_fmaf(a.w, b.w, base);
                    acc = hw_fmaf(ea.x, eb.x, acc);
                    acc = hw_fmaf(ea.y, eb.y, acc);
                    acc = hw_fmaf(ea.z, eb.z, acc);
                    acc = hw_fmaf(ea.w, eb.w, acc);
                }
                if (g0 + kQuadGroup <= NB) {
                    row(QR_D + 1 + u)[0] = ownD[kQuadGroup];
                    if (u == 0) row(QR_D)[0] = row(QR_D)[kQuadGroup];
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
            // The last boundary's own terms: its weight is that of the bin before it.
            {
                constexpr int kLastThread = NB % kQuadGroup / kRecurBlock;
                const float F = cLast == NB ? EmQuadAt<kLastThread>(fFirst) : fC;
                const float x = h.Start(cLast);
                const float G = x * F, dev = x - piv;
                const float dOwn = ownD[at], dBl = row(QR_D)[at];
                const float w = dBl * F;
                own = hw_fmaf(dOwn, F, own);
                ownX = hw_fmaf(dOwn, G, ownX);
                base = hw_fmaf(u < 2 ? dBl : u == 2 ? w : w * dev, u == 0 ? F : u == 1 ? G : dev, base);
            }
            ci[0] = EmQuadAt<0>(base);
            mom1[0] = EmQuadAt<1>(base);
            q1 = EmQuadAt<2>(base);
            q2 = EmQuadAt<3>(base);
            ci[1] = EmQuadAt<0>(own);
            ci[2] = EmQuadAt<1>(own);
            ci[3] = EmQuadAt<2>(own);
            ci[4] = EmQuadAt<3>(own);
            mom1[1] = EmQuadAt<0>(ownX);
            mom1[2] = EmQuadAt<1>(ownX);
            mom1[3] = EmQuadAt<2>(ownX);
            mom1[4] = EmQuadAt<3>(ownX);
            probSum = EmQuadAt<0>(acc);
            wps = EmQuadAt<1>(acc);
        } else {
        uint32_t exMask = 0;   // this ZMW's components that take exp at every boundary of the block
        uint32_t exAny = 0;    // the same for any ZMW of the wave
        bool zeroBl = false;   // the baseline density is +0 through the block for the whole wave
        auto restart = [&](int c, auto expOf) {
            const float x0 = h.Start(c);
            float dl[5];
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                const float y0 = x0 - mu[i];
                const float t0 = hw_fmaf(y0 * y0, nhv[i], pref[i]);
                // t(x0 + bs) - t(x0) on the ideal grid (no cancellation of rounded t)
                dl[i] = nbs[i] * hw_fmaf(2.0f, y0, h.bs);
                // exp(t) is +0 below the threshold: waves skip the exp when all ZMWs are, and
                // then the ratio's too.  The density stays +0 through the block (+0 times any
                // finite ratio >= 0); a rising one (dl > 0) takes exp at every boundary below.
                const bool zero = __all(t0 < kExpZeroBelow);
                if (i == 0) zeroBl = zero;
                if (zero) {
                    dd[i] = 0.0f;
                    rr[i] = 0.0f;
                } else {
                    dd[i] = expOf(t0);
                    rr[i] = expOf(dl[i]);
                }
            }
            // No ZMW leaves the recurrence when every density is at least FLT_MIN or falling
            // (max(dd, -dl) >= FLT_MIN) and no ratio is above e^80; the comparisons are false
            // for NaN, which takes the exact test.
            float lo = __builtin_fmaxf(dd[0], -dl[0]), hi = dl[0];
#pragma unroll
            for (int i = 1; i < 5; ++i) {
                lo = __builtin_fminf(lo, __builtin_fmaxf(dd[i], -dl[i]));
                hi = __builtin_fmaxf(hi, dl[i]);
            }
            exMask = 0;
            exAny = 0;
            if (!bounded || !__all(lo >= FLT_MIN && hi <= 80.0f)) {
                // A component that starts the block below the zero threshold and is still
                // below it, and still left of its mean, at the block's end has +0 for every
                // exp in between (t rises up to the mean; the threshold leaves a margin of 1
                // for its rounding): the recurrence from +0 gives the same, with a ratio of 0.
                const float x1 = h.Start(c + kRecurBlock);
#pragma unroll
                for (int i = 0; i < 5; ++i) {
                    const bool rec = (dd[i] >= FLT_MIN || dl[i] <= 0.0f) && dl[i] <= 80.0f;
                    const bool flat = tAt(x0, i) < kExpZeroBelow && tAt(x1, i) < kExpZeroBelow && x1 <= mu[i];
                    if (!rec && flat) rr[i] = 0.0f;   // (never for a NaN density)
                    const bool ex = !rec && !flat && ((nanComp >> i) & 1u) == 0u;
                    exMask |= (ex ? 1u : 0u) << i;
                    exAny |= (__any(ex) ? 1u : 0u) << i;
                }
                exAny = __builtin_amdgcn_readfirstlane(exAny);
                zeroBl = zeroBl && (exAny & 1u) == 0u;
            }
        };
        // One boundary c with densities dd and the count n of the bin before it: that bin's
        // probability, its term of the log-likelihood and f = n / binp, then the sums of
        // boundary c - 1 with weight F = f_{c-2} + f_{c-1}.  Where the wave's counts are all
        // zero the terms are exact zeros (every density is finite) and may be left out.
        float bpPrev = 0.0f, fPrev = 0.0f, dPrev[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        auto binProb = [&](int c, bool bl) {
            const float a0 = bl ? dd[0] + dd[1] : dd[1];
            const float bp = a0 + (dd[2] + (dd[3] + dd[4]));   // Sum5Tree
            // binp >= binProbMin >= FLT_MIN and finite: the log needs no special cases
            const float binp = hw_max_pos(halfBin * (bpPrev + bp), binProbMin);
            probSum = c == 0 ? 0.0f : probSum + binp;   // (there is no bin before boundary 0)
            bpPrev = bp;
            return binp;
        };
        auto weigh = [&](float binp, uint32_t n) {
            const float nj = (float)n;
            float lg, rcp;
            hw_log_rcp_tab(binp, sRc, sLc, &lg, &rcp);
            wps = hw_fmaf(nj, lg, wps);
            return nj * rcp;
        };
        auto gather = [&](float x, float F, bool bl) {
            const float G = x * F;
#pragma unroll
            for (int m = bl ? 0 : 1; m < 5; ++m) {
                ci[m] = hw_fmaf(dPrev[m], F, ci[m]);
                mom1[m] = hw_fmaf(dPrev[m], G, mom1[m]);
            }
            if (bl) {
                const float dev = x - piv;
                const float w = dPrev[0] * F;
                q1 = hw_fmaf(w, dev, q1);
                q2 = hw_fmaf(w * dev, dev, q2);
            }
        };
        auto keep = [&]() {
#pragma unroll
            for (int m = 0; m < 5; ++m) dPrev[m] = dd[m];
        };
        auto advance = [&](bool bl) {
#pragma unroll
            for (int i = bl ? 0 : 1; i < 5; ++i) {
                dd[i] = dd[i] * rr[i];
                rr[i] = rr[i] * qq[i];
            }
        };
        // The tail of the histogram is left out once, for every ZMW of the wave, the bins
        // ahead are empty, the boundary lies beyond every mode's mean (so each density
        // only falls from here on) and bs times the density sum is below 2^-27 of
        // probSum, as is binProbMin: then every remaining bin probability is below half
        // an ulp of probSum, so adding them would leave it unchanged, and every other sum
        // of those boundaries is an exact zero (empty bins).  The result equals the full
        // pass bit for bit.
        // Counts of a block's bins b0 - 1 .. b0 + 8, each read again for the next block as
        // soon as it has been used, so its load is in flight over a whole block.
        uint32_t cn[kRecurBlock];
#pragma unroll
        for (int j = 0; j < kRecurBlock; ++j) cn[j] = (j == 0) ? 0u : h.Cnt(j - 1);
        int cLast = NB;   // the last boundary taken
#pragma unroll 1
        for (int b0 = 0; b0 <= NB; b0 += kRecurBlock) {
            if (b0 > 0) {
                const float tol = hw_ldexpf(probSum, -27);
                const bool tail = lastNz < b0 - 1 && h.Start(b0 - 1) > maxMu && h.bs * bpPrev < tol && binProbMin < tol;
                if (__all(tail)) {
                    cLast = b0 - 1;
                    break;
                }
            }
            if (bounded) restart(b0, [](float t) { return ExpBounded(t); });
            else restart(b0, [](float t) { return hw_expf(t); });
            if (b0 == NB) {   // the last boundary: bin NB - 1
                const float f = weigh(binProb(NB, true), h.Cnt(NB - 1));
                gather(h.Start(NB - 1), fPrev + f, true);
                fPrev = f;
                keep();
                break;
            }
            uint32_t none = 0;   // bins empty for the whole wave
#pragma unroll
            for (int j = 0; j < kRecurBlock; ++j) none |= (__all(cn[j] == 0u) ? 1u : 0u) << j;
            none = __builtin_amdgcn_readfirstlane(none);
            // Row of the next block's first bin (the last block's own is read when it is needed).
            const uint16_t* ahead = &h.h->bin_count[min(b0 + kRecurBlock - 1, NB - kRecurBlock)][zin];
            if (exAny != 0u || __popc(none) > 1) {
                // Some component takes exp at every boundary, or bins are empty for the whole
                // wave: both are left to wave-uniform branches.
                bool noF = __all(fPrev == 0.0f);
#pragma unroll
                for (int j = 0; j < kRecurBlock; ++j) {
                    if (j > 0) {
                        advance(true);
                        if (exAny != 0u) {
                            const float x = h.Start(b0 + j);
#pragma unroll
                            for (int i = 0; i < 5; ++i) {
                                if ((exAny >> i) & 1u) {
                                    const float v = hw_expf(tAt(x, i));
                                    dd[i] = ((exMask >> i) & 1u) ? v : dd[i];
                                }
                            }
                        }
                    }
                    const float binp = binProb(b0 + j, true);
                    const bool empty = (none >> j) & 1u;
                    if (!(empty && noF)) {
                        const float f = empty ? 0.0f : weigh(binp, cn[j]);
                        gather(h.Start(b0 + j - 1), fPrev + f, true);
                        fPrev = f;
                    }
                    noF = empty;
                    keep();
                    cn[j] = ahead[j * LS];
                }
            } else if (zeroBl) {
#pragma unroll
                for (int j = 0; j < kRecurBlock; ++j) {
                    if (j > 0) advance(false);
                    const float f = weigh(binProb(b0 + j, false), cn[j]);
                    gather(h.Start(b0 + j - 1), fPrev + f, j == 0);
                    fPrev = f;
                    keep();
                    cn[j] = ahead[j * LS];
                }
            } else {
#pragma unroll
                for (int j = 0; j < kRecurBlock; ++j) {
                    if (j > 0) advance(true);
                    const float f = weigh(binProb(b0 + j, true), cn[j]);
                    gather(h.Start(b0 + j - 1), fPrev + f, true);
                    fPrev = f;
                    keep();
                    cn[j] = ahead[j * LS];
                }
            }
        }
        gather(h.Start(cLast), fPrev, true);
        }
        const float q0 = ci[0];
#pragma unroll
        for (int m = 0; m < 5; ++m) {
            ci[m] *= halfBin;
            mom1[m] *= halfBin;
        }
        const float logLikePrev = logLike;
        logLike = wps - njSum * hw_cephes_logf(probSum);
        const float ds = s - sExpect;
        logLike -= 0.5f * (ds * ds) * sExpectWeight;
        const float delta = logLike - logLikePrev;
        const float convTol = (MODE == EM_LEARNED ? x.convTol : 1e-4f) * hw_fabsf(logLike);
        bool conv = (delta >= 0.0f) && (delta < convTol);
        conv = conv && (logLike >= mlLogLike);
        if (conv) {
            mlLogLike = logLike;
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                rhoEst[k] = rho[k];
                muEst[k] = mu[k];
                varEst[k] = var[k];
            }
        }
        converged = converged || conv;
        // Lane-wide early exit (DmeEmHost.cpp:485)
        const bool done = converged || (status != HWPA_ZS_OK) || gated;
        if (!d.iterToLimit && laneAll(done)) break;

        // ---- M-step
        float c[5];
#pragma unroll
        for (int m = 0; m < 5; ++m) c[m] = hw_maxf(ci[m], 0.1f);
#pragma unroll
        for (int m = 0; m < 5; ++m) rho[m] = c[m] / njSum;
        {
            const float rs = Sum5Tree(rho);
#pragma unroll
            for (int m = 0; m < 5; ++m) rho[m] = rho[m] / rs;
        }
        mu[0] = mom1[0] / c[0];
        float numer = 0.0f, denom = 0.0f;
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            const int i = a + 1;
            numer += rpa[a] * varinv[i] * mom1[i];
            denom += (rpa[a] * rpa[a]) * varinv[i] * c[i];
        }
        numer += sExpect * sExpectWeight;
        denom += sExpectWeight;
        s = numer / denom;
        const float minPulseMean = hw_maxf(1.0f, d.signalScaler);
        const float sMin = hw_maxf(0.5f * hw_sqrtf(var[0]), minPulseMean) / rpaMin;
        if (s < sMin) {
            s = sMin;
            status |= HWPA_ZS_VLOW_SIGNAL;
        }
#pragma unroll
        for (int a = 0; a < NA; ++a) mu[a + 1] = s * rpa[a];
        // Baseline second moment about the new mean, from the moments about piv.
        const float dl = mu[0] - piv;
        float mom2 = (q2 - (2.0f * dl) * q1) + (dl * dl) * q0;
        mom2 *= 0.5f * h.bs;
        var[0] = mom2 / c[0] + varQuant;
        var[0] = hw_clampf(var[0], d.blVarMin, d.blVarMax);
#pragma unroll
        for (int a = 0; a < NA; ++a) var[a + 1] = Covar(d, d.cv[a] * d.cv[a], mu[a + 1], var[0]);
    }
    if (!converged) status |= HWPA_ZS_NO_CONVERGE;
    if (threadIdx.x == 0 && iters) iters[lane] = it;

    work.bl.w = rhoEst[0];
    work.bl.mean = muEst[0];
    work.bl.var = varEst[0];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        work.an[a].w = rhoEst[a + 1];
        work.an[a].mean = muEst[a + 1];
        work.an[a].var = varEst[a + 1];
    }

    // ComputeConfidence (DmeEmHost.cpp:717-803); the G-test factor stays 1.
    float conf = 1.0f;
    {
        float cf[8];
        cf[0] = converged ? 1.0f : 0.0f;
        cf[1] = hw_satlin(0.05f, 0.15f, work.bl.w);
        float x = (work.bl.mean * work.bl.mean) / work.bl.var;
        cf[2] = hw_cephes_expf(-x / (2.0f * (1.0f * 1.0f)));
        x = hw_dlog2f(work.bl.var / det.bl.var);
        const float tol = 1.5f / (0.5f + det.conf);
        cf[3] = hw_cephes_expf(-x * x / (2.0f * (tol * tol)));
        x = 1.0f;
        if (d.mixThresh1 > 0.0f) {
            x *= hw_satlin(d.mixThresh0, d.mixThresh1, work.an[0].w);
            x *= hw_satlin(d.mixThresh0, d.mixThresh1, work.an[NA - 1].w);
        }
        cf[4] = x;
        const float bgSigma = hw_sqrtf(work.bl.var);
        x = work.an[NA - 1].mean;
        x /= bgSigma;
        cf[5] = hw_satlin(d.snrThresh0, d.snrThresh1, x);
        if (d.snrDrop < 0.0f) {
            cf[6] = 1.0f;
        } else {
            const float snrEst = work.an[0].mean / bgSigma;
            const float refBgSigma = hw_sqrtf(det.bl.var);
            const float refSnr0 = det.an[0].mean / refBgSigma;
            float refSnr1 = det.an[1].mean / refBgSigma;
            refSnr1 *= d.snrDrop;
            refSnr1 *= hw_minf(det.conf, 1.0f);
            cf[6] = hw_satlin(refSnr1, hw_sqrtf(refSnr0 * refSnr1), snrEst);
        }
        cf[7] = 1.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) conf *= cf[k];
    }
    conf = hw_minf(hw_maxf(0.0f, conf), 1.0f);
    conf = (conf >= d.successThresh) ? conf : 0.0f;
    if (x.diag && u == 0) {
        float* dg = x.diag + (size_t)lane * HWPA_EM_DIAG_ROWS * LS + z;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            dg[k * LS] = rhoEst[k];
            dg[(5 + k) * LS] = muEst[k];
            dg[(10 + k) * LS] = varEst[k];
        }
        dg[15 * LS] = conf;
        dg[16 * LS] = converged ? 1.0f : 0.0f;
        dg[17 * LS] = (float)status;
    }
    if (MODE == EM_LEARNED) {
        const bool accept = !gated && converged && status == HWPA_ZS_OK && conf >= x.acceptConf;
        if (u == 0) x.fallback[(size_t)lane * LS + z] = accept ? 0 : 1;
        if (!accept) return;
    }
    work.conf = conf;
    UpdateConf(d, det, work);
    if (zin == z && u == 0) StoreModel(det, lm, z);
}

// ---- fallback compaction for the learned start ---------------------------------
// A lane whose 64 ZMWs were all rejected runs the plain EM in place.  The
// rejected ZMWs of the other lanes are packed densely (in lane order, so the
// grouping is deterministic) into compact lanes, run through the plain EM and
// scattered back.

__device__ __forceinline__ void ColStatAcc(const hwpa_stat_acc& s, hwpa_stat_acc& d, int sz, int dz)
{
    d.offset[dz] = s.offset[sz];
    d.m0[dz] = s.m0[sz];
    d.m1[dz] = s.m1[sz];
    d.m2[dz] = s.m2[sz];
}

__device__ void ColStats(const hwpa_baseliner_stats& s, hwpa_baseliner_stats& d, int sz, int dz)
{
    ColStatAcc(s.full.basic, d.full.basic, sz, dz);
    d.full.lag_m2[dz] = s.full.lag_m2[sz];
    for (int k = 0; k < HWPA_AUTOCORR_LAG; ++k) {
        d.full.fbuf[k][dz] = s.full.fbuf[k][sz];
        d.full.bbuf[k][dz] = s.full.bbuf[k][sz];
    }
    d.full.bidx[0][dz] = s.full.bidx[0][sz];
    d.full.bidx[1][dz] = s.full.bidx[1][sz];
    d.trace_min[dz] = s.trace_min[sz];
    d.trace_max[dz] = s.trace_max[sz];
    ColStatAcc(s.baseline, d.baseline, sz, dz);
    d.raw_baseline_sum[dz] = s.raw_baseline_sum[sz];
    ColStatAcc(s.background, d.background, sz, dz);
}

__device__ void ColModel(const hwpa_lane_model& s, hwpa_lane_model& d, int sz, int dz)
{
    for (int a = 0; a < NA; ++a) {
        d.analogs[a].means[dz] = s.analogs[a].means[sz];
        d.analogs[a].vars[dz] = s.analogs[a].vars[sz];
        d.analogs[a].weights[dz] = s.analogs[a].weights[sz];
    }
    d.baseline.means[dz] = s.baseline.means[sz];
    d.baseline.vars[dz] = s.baseline.vars[sz];
    d.baseline.weights[dz] = s.baseline.weights[sz];
    d.confidence[dz] = s.confidence[sz];
}

__global__ __launch_bounds__(64) void FallbackCountKernel(const uint8_t* __restrict__ fb, uint32_t* __restrict__ cnt)
{
    const uint64_t m = __ballot(fb[(size_t)blockIdx.x * LS + threadIdx.x] != 0);
    if (threadIdx.x == 0) cnt[blockIdx.x] = (uint32_t)__popcll(m);
}

// Exclusive scan of per-lane counts in one workgroup (fixed order).  Lanes whose
// 64 ZMWs all fall back run the plain EM in place and take no compact slots:
// total[0] counts the compacted ZMWs, total[1] every fallback ZMW.
__global__ __launch_bounds__(1024) void FallbackScanKernel(const uint32_t* __restrict__ cnt, uint32_t lanes,
                                                           uint32_t* __restrict__ off, uint32_t* __restrict__ total)
{
    __shared__ uint32_t part[16], whole[16];
    const uint32_t per = (lanes + 1023) / 1024;
    const uint32_t b0 = threadIdx.x * per, b1 = min(lanes, b0 + per);
    uint32_t s = 0, w = 0;
    for (uint32_t i = b0; i < b1; ++i) {
        const uint32_t c = cnt[i];
        s += c == LS ? 0u : c;
        w += c == LS ? c : 0u;
    }
    // Inclusive sums over the wave, then over the 16 waves.
    const uint32_t t = threadIdx.x % 64, wv = threadIdx.x / 64;
    uint32_t incl = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d, 64);
        if (t >= (uint32_t)d) incl += y;
        w += __shfl_xor(w, d, 64);
    }
    if (t == 63) {
        part[wv] = incl;
        whole[wv] = w;
    }
    __syncthreads();
    uint32_t before = 0, sum = 0, all = 0;
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) {
        before += k < wv ? part[k] : 0u;
        sum += part[k];
        all += whole[k];
    }
    if (threadIdx.x == 0) {
        total[0] = sum;
        total[1] = sum + all;
    }
    uint32_t run = before + incl - s;
    for (uint32_t i = b0; i < b1; ++i) {
        off[i] = run;
        const uint32_t c = cnt[i];
        run += c == LS ? 0u : c;
    }
}

// One workgroup per lane: its four waves share the lane's bins, read 15 at a time (one wave
// copying bin after bin took 75 us for 4,096 lanes, these 70: the rest is the traffic, rows
// written in parts).
constexpr int kGatherBatch = 15;
static_assert(NB % (4 * kGatherBatch) == 0, "whole batches per wave");

__global__ __launch_bounds__(256) void FallbackGatherKernel(const uint8_t* __restrict__ fb, const uint32_t* __restrict__ off,
                                                            const hwpa_lane_hist* __restrict__ hist,
                                                            const hwpa_baseliner_stats* __restrict__ stats,
                                                            const hwpa_lane_model* __restrict__ models,
                                                            hwpa_lane_hist* cHist, hwpa_baseliner_stats* cStats,
                                                            hwpa_lane_model* cModels, uint32_t* __restrict__ map)
{
    const int lane = blockIdx.x, z = threadIdx.x % LS, w = threadIdx.x / LS;
    const bool f = fb[(size_t)lane * LS + z] != 0;
    const uint64_t m = __ballot(f);
    if (!f || m == ~0ull) return;
    const uint32_t rank = (uint32_t)__popcll(m & ((1ull << z) - 1ull));
    const uint32_t pos = off[lane] + rank;
    const uint32_t cl = pos / LS;
    const int dz = (int)(pos % LS);
    const hwpa_lane_hist& s = hist[lane];
    hwpa_lane_hist& d = cHist[cl];
    for (int b = w * (NB / 4); b < (w + 1) * (NB / 4); b += kGatherBatch) {
        uint16_t c[kGatherBatch];
#pragma unroll
        for (int j = 0; j < kGatherBatch; ++j) c[j] = s.bin_count[b + j][z];
#pragma unroll
        for (int j = 0; j < kGatherBatch; ++j) d.bin_count[b + j][dz] = c[j];
    }
    if (w == 0) {
        d.low_bound[dz] = s.low_bound[z];
        d.bin_size[dz] = s.bin_size[z];
        d.outlier_low[dz] = s.outlier_low[z];
        d.outlier_high[dz] = s.outlier_high[z];
        map[pos] = (uint32_t)lane * LS + (uint32_t)z;
    } else if (w == 1) {
        ColStats(stats[lane], cStats[cl], z, dz);
    } else if (w == 2) {
        ColModel(models[lane], cModels[cl], z, dz);
    }
}

__global__ __launch_bounds__(64) void FallbackScatterKernel(const uint32_t* __restrict__ total,
                                                            const uint32_t* __restrict__ map,
                                                            const hwpa_lane_model* __restrict__ cModels,
                                                            hwpa_lane_model* models)
{
    const uint32_t pos = blockIdx.x * LS + threadIdx.x;
    if (pos >= *total) return;
    const uint32_t dst = map[pos];
    ColModel(cModels[blockIdx.x], models[dst / LS], (int)threadIdx.x, (int)(dst % LS));
}

int32_t DmeInitModels(const hwpa_config& cfg, const hwpa_baseliner_stats* stats, hwpa_lane_model* models,
                      uint32_t lanes, hipStream_t s)
{
    if (!stats || !models || lanes == 0) return Fail(HWPA_ERR_INVALID_ARG, "dme_init_models: bad argument");
    hipLaunchKernelGGL(DmeInitKernel, dim3(lanes), dim3(LS), 0, s, stats, models, MakeDevCfg(cfg));
    return CheckLaunch("DmeInitKernel");
}

// DmeEmHost::EvolveModel (DmeEmHost.cpp:806-834), DetectionModelHost::EvolveConfidence
static float EvolveFactor(const DmeDevCfg& d, const int32_t model_fi[2], const int32_t est_fi[2])
{
    const int32_t tModel = model_fi[0] + (int32_t)((uint32_t)(model_fi[1] - model_fi[0]) / 2u);
    const int32_t tEst = est_fi[0] + (int32_t)((uint32_t)(est_fi[1] - est_fi[0]) / 2u);
    const float thl = 0.5f * (float)(tModel + tEst);
    const float hl = d.hl0 + (d.hl1 - d.hl0) * hw_satlin(56160.0f, 168480.0f, thl);
    const float tDiff = (float)(tEst - tModel);
    return hw_dexp2f(-hw_fabsf(tDiff) / hl);
}

// Up to one lane per CU, four threads per ZMW (the kernel's QUAD form; its rows take 143 KB of
// LDS, so a second lane on the CU waits for the first).
constexpr uint32_t kEmQuadLanes = 256;

// Waves per SIMD for a launch of `lanes` lanes on 1,024 SIMDs (1: four threads per ZMW).  Lanes
// take about equally long, so what counts is the number of rounds.  Up to 2,048 lanes two waves per
// SIMD are all there are, and the registers of 2 spill nothing (2,048 lanes, start-up estimate:
// 1.47 ms; held to 3 waves 1.59, to 4 1.87); 3,073 to 4,096 lanes fit one round of 4 (4,096: 2.68
// ms; 3 waves, whose second round is a third full, 3.03); beyond, 3 is the best (32,768 lanes in a
// running pool: 12.7 ms; 4 13.2, 2 15.0; 8,192: 4.99; 5.35, 5.53), and between 2,049 and 3,072 its
// round suffices.  Pools that run side by side share the SIMDs (sideBySide, their lanes together):
// there a launch with fewer waves per SIMD keeps others out, and 3 is the choice past 2,048 (six
// pools of 365 to 2,048 lanes in one graph: 7.1 ms a step, 7.5 with each pool's own choice; three
// pools of 2,000 lanes on their streams: 1.71 ms a chunk against 1.82).  Analyzers always pass a count of
// lanes, so 4 serves estimates without one.  Four threads per ZMW pay up to three pools of 256
// lanes, which is what the hardware queues let run at a time (a chunk with them and with one thread,
// us, for one, two, three, four, six and eight pools of 200 lanes: 1051, 625, 536, 659, 550, 585 and
// 1425, 810, 563, 784, 566, 616; of 256 lanes: 1057, 783, 579, 706, 681, 670 and 1434, 825, 641, 838,
// 644, 703).
static int EmWavesPerSimd(uint32_t lanes, uint32_t sideBySide)
{
    constexpr uint32_t kSimds = 1024;
    const uint32_t all = std::max(lanes, sideBySide);
    if (lanes <= kEmQuadLanes && all <= 3 * kEmQuadLanes) return 1;
    if (all <= 2 * kSimds) return 2;
    return (sideBySide == 0 && lanes > 3 * kSimds && lanes <= 4 * kSimds) ? 4 : 3;
}

template <int MODE>
static int32_t EmLaunch(int waves, uint32_t lanes, hipStream_t s, const hwpa_lane_hist* hist,
                        const hwpa_baseliner_stats* stats, hwpa_lane_model* models, int32_t* iters, const DmeDevCfg& d,
                        float evolve, const EmExtra& x)
{
    if (waves == 1) {
        hipLaunchKernelGGL((DmeEstimateKernel<MODE, 1, true>), dim3(lanes), dim3(4 * LS), 0, s, hist, stats, models,
                           iters, d, evolve, x);
        return CheckLaunch("DmeEstimateKernel");
    }
#define HWPA_EM_LAUNCH(W)                                                                                             \
    hipLaunchKernelGGL((DmeEstimateKernel<MODE, W>), dim3(lanes), dim3(LS), 0, s, hist, stats, models, iters, d, evolve, x)
    switch (waves) {
    case 2: HWPA_EM_LAUNCH(2); break;
    case 4: HWPA_EM_LAUNCH(4); break;
    default: HWPA_EM_LAUNCH(3); break;
    }
#undef HWPA_EM_LAUNCH
    return CheckLaunch("DmeEstimateKernel");
}

int32_t DmeEstimate(const hwpa_config& cfg, const hwpa_lane_hist* hist, const hwpa_baseliner_stats* stats,
                    hwpa_lane_model* models, const int32_t model_fi[2], const int32_t est_fi[2], uint32_t lanes,
                    int32_t* d_iters, hipStream_t s, float* diag, uint32_t sideBySide)
{
    if (!hist || !stats || !models || lanes == 0) return Fail(HWPA_ERR_INVALID_ARG, "dme_estimate: bad argument");
    const DmeDevCfg d = MakeDevCfg(cfg);
    const float evolve = EvolveFactor(d, model_fi, est_fi);
    EmExtra x{};
    x.diag = diag;
    return EmLaunch<EM_PLAIN>(EmWavesPerSimd(lanes, sideBySide), lanes, s, hist, stats, models, d_iters, d, evolve, x);
}

void LearnedWsFree(LearnedWs& w)
{
    DeviceFree(w.y);
    DeviceFree(w.fallback);
    DeviceFree(w.cnt);
    DeviceFree(w.off);
    DeviceFree(w.total);
    DeviceFree(w.map);
    DeviceFree(w.cHist);
    DeviceFree(w.cStats);
    DeviceFree(w.cModels);
    DeviceFree(w.cIters);
    w = LearnedWs{};
}

int32_t LearnedWsAlloc(LearnedWs& w, uint32_t lanes)
{
    LearnedWsFree(w);
    const size_t Z = (size_t)lanes * LS;
    struct {
        void** p;
        size_t n;
    } req[] = {
        {(void**)&w.y, Z * HWPA_MLP_OUT * 4},
        {(void**)&w.fallback, Z},                 {(void**)&w.cnt, (size_t)lanes * 4},
        {(void**)&w.off, (size_t)lanes * 4},      {(void**)&w.total, 16},
        {(void**)&w.map, Z * 4},                  {(void**)&w.cHist, (size_t)lanes * sizeof(hwpa_lane_hist)},
        {(void**)&w.cStats, (size_t)lanes * sizeof(hwpa_baseliner_stats)},
        {(void**)&w.cModels, (size_t)lanes * sizeof(hwpa_lane_model)}, {(void**)&w.cIters, (size_t)lanes * 4},
    };
    for (auto& r : req) {
        const int32_t rc = DeviceAlloc(r.p, r.n, "learned-start workspace");
        if (rc != HWPA_OK) {
            LearnedWsFree(w);
            return rc;
        }
    }
    w.lanes = lanes;
    return HWPA_OK;
}

int32_t DmeEstimateLearned(const hwpa_config& cfg, hwpa_initializer* mlp, LearnedWs& w, const hwpa_lane_hist* hist,
                           const hwpa_baseliner_stats* stats, hwpa_lane_model* models, const int32_t model_fi[2],
                           const int32_t est_fi[2], uint32_t lanes, int32_t* d_iters, hipStream_t s,
                           uint32_t sideBySide)
{
    if (!mlp || !hist || !stats || !models || lanes == 0 || lanes > w.lanes)
        return Fail(HWPA_ERR_INVALID_ARG, "dme_estimate_learned: bad argument");
    if (cfg.learned_em_iteration_limit == 0) return Fail(HWPA_ERR_BAD_CONFIG, "learned EM iteration limit must be positive");
    const DmeDevCfg d = MakeDevCfg(cfg);
    const float evolve = EvolveFactor(d, model_fi, est_fi);
    int32_t rc = MlpForwardFromHist(mlp, hist, lanes, w.y, s);
    if (rc != HWPA_OK) return rc;
    EmExtra x{};
    x.init = w.y;
    x.omap = MlpOutputMap(mlp);
    x.fallback = w.fallback;
    x.acceptConf = cfg.learned_conf_threshold;
    x.convTol = cfg.learned_conv_tol;
    x.iterLimit = (int32_t)cfg.learned_em_iteration_limit;
    x.gateLogit = MlpGateLogit(cfg.learned_gate_threshold);
    x.laneMinConf = (int32_t)cfg.learned_lane_min_confident;
    const int waves = EmWavesPerSimd(lanes, sideBySide);
    if ((rc = EmLaunch<EM_LEARNED>(waves, lanes, s, hist, stats, models, d_iters, d, evolve, x)) != HWPA_OK) return rc;
    hipLaunchKernelGGL(FallbackCountKernel, dim3(lanes), dim3(LS), 0, s, w.fallback, w.cnt);
    if ((rc = CheckLaunch("FallbackCountKernel")) != HWPA_OK) return rc;
    hipLaunchKernelGGL(FallbackScanKernel, dim3(1), dim3(1024), 0, s, w.cnt, lanes, w.off, w.total);
    if ((rc = CheckLaunch("FallbackScanKernel")) != HWPA_OK) return rc;
    hipLaunchKernelGGL(FallbackGatherKernel, dim3(lanes), dim3(4 * LS), 0, s, w.fallback, w.off, hist, stats, models,
                       w.cHist, w.cStats, w.cModels, w.map);
    if ((rc = CheckLaunch("FallbackGatherKernel")) != HWPA_OK) return rc;
    EmExtra q{};
    q.laneSel = w.fallback;
    if ((rc = EmLaunch<EM_PLAIN>(waves, lanes, s, hist, stats, models, nullptr, d, evolve, q)) != HWPA_OK) return rc;
    // How many of these lanes have work is known on the device only; it is seldom all of them.
    // Up to kEmQuadLanes of them are estimated by four threads per ZMW, so past that size, unless
    // other pools need the SIMDs, two launches go out of which one has work (the other's waves end
    // at once, 5 us).  300 lanes, over half of their ZMWs rejected: 1.21 ms, one launch 1.78.
    EmExtra p{};
    p.active = w.total;
    p.activeMax = UINT32_MAX;
    if (lanes > kEmQuadLanes && sideBySide <= 3ull * lanes) {
        p.activeMax = kEmQuadLanes * (uint32_t)LS;
        rc = EmLaunch<EM_PLAIN>(1, kEmQuadLanes, s, w.cHist, w.cStats, w.cModels, w.cIters, d, evolve, p);
        if (rc != HWPA_OK) return rc;
        p.activeMin = p.activeMax + 1;
        p.activeMax = UINT32_MAX;
    }
    rc = EmLaunch<EM_PLAIN>(std::min(waves, 3), lanes, s, w.cHist, w.cStats, w.cModels, w.cIters, d, evolve, p);
    if (rc != HWPA_OK) return rc;
    hipLaunchKernelGGL(FallbackScatterKernel, dim3(lanes), dim3(LS), 0, s, w.total, w.map, w.cModels, models);
    return CheckLaunch("FallbackScatterKernel");
}

}  // namespace hwpa

// ---- learned-start estimation without allocation ---------------------------
// The workspace of DmeEstimateLearned for at most HWPA_NOALLOC_MAX_LANES lanes,
// in one device array.  Host code never passes `scratch` itself to a kernel
// (its host-side name is not a device address): NoAllocScratch looks the
// array's device address up once per device with hipGetSymbolAddress.
// Every buffer carved from it is written before it is read within one call,
// so nothing needs clearing between calls.

namespace hwpa {

constexpr size_t kNoAllocAlign = 256;
constexpr size_t AlignUp(size_t n) { return (n + kNoAllocAlign - 1) / kNoAllocAlign * kNoAllocAlign; }

// Bytes of the learned-start workspace for `lanes` lanes, each buffer
// starting on a 256-byte boundary (the order of CarveLearnedWs).
constexpr size_t LearnedWsBytes(size_t lanes)
{
    return AlignUp(lanes * LS * HWPA_MLP_OUT * 4) + AlignUp(lanes * LS) + AlignUp(lanes * 4) + AlignUp(lanes * 4) +
           AlignUp(16) + AlignUp(lanes * LS * 4) + AlignUp(lanes * sizeof(hwpa_lane_hist)) +
           AlignUp(lanes * sizeof(hwpa_baseliner_stats)) + AlignUp(lanes * sizeof(hwpa_lane_model)) +
           AlignUp(lanes * 4);
}

constexpr size_t kNoAllocBytes = LearnedWsBytes(HWPA_NOALLOC_MAX_LANES);

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocMaxDevices = 64;

static int32_t NoAllocScratch(unsigned char** out)
{
    static std::mutex mu;
    static void* addr[kNoAllocMaxDevices] = {};
    int dev = -1;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return Fail(HWPA_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
    if (dev < 0 || dev >= kNoAllocMaxDevices) return Fail(HWPA_ERR_UNSUPPORTED, "device index beyond the workspace table");
    std::lock_guard<std::mutex> g(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        const hipError_t r = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (r != hipSuccess || !p)
            return Fail(HWPA_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(r));
        addr[dev] = p;
    }
    *out = static_cast<unsigned char*>(addr[dev]);
    return HWPA_OK;
}

static LearnedWs CarveLearnedWs(unsigned char* base, uint32_t lanes)
{
    LearnedWs w{};
    size_t at = 0;
    auto take = [&](size_t n) {
        unsigned char* p = base + at;
        at += AlignUp(n);
        return p;
    };
    const size_t L = lanes;
    w.y = reinterpret_cast<float*>(take(L * LS * HWPA_MLP_OUT * 4));
    w.fallback = take(L * LS);
    w.cnt = reinterpret_cast<uint32_t*>(take(L * 4));
    w.off = reinterpret_cast<uint32_t*>(take(L * 4));
    w.total = reinterpret_cast<uint32_t*>(take(16));
    w.map = reinterpret_cast<uint32_t*>(take(L * LS * 4));
    w.cHist = reinterpret_cast<hwpa_lane_hist*>(take(L * sizeof(hwpa_lane_hist)));
    w.cStats = reinterpret_cast<hwpa_baseliner_stats*>(take(L * sizeof(hwpa_baseliner_stats)));
    w.cModels = reinterpret_cast<hwpa_lane_model*>(take(L * sizeof(hwpa_lane_model)));
    w.cIters = reinterpret_cast<int32_t*>(take(L * 4));
    w.lanes = lanes;
    return w;
}

}  // namespace hwpa

extern "C" int32_t hwpa_dme_estimate_learned_noalloc(const hwpa_config* cfg, hwpa_initializer* m,
                                                     const hwpa_lane_hist* d_hist,
                                                     const hwpa_baseliner_stats* d_stats, hwpa_lane_model* d_models,
                                                     const int32_t model_fi[2], const int32_t est_fi[2],
                                                     uint32_t lanes, int32_t* d_iters, uint32_t* fallback_count,
                                                     void* stream)
{
    using namespace hwpa;
    if (!cfg || !m || !model_fi || !est_fi || lanes == 0)
        return Fail(HWPA_ERR_INVALID_ARG, "dme_estimate_learned_noalloc: null argument or no lanes");
    if (lanes > HWPA_NOALLOC_MAX_LANES)
        return Fail(HWPA_ERR_INVALID_ARG, "dme_estimate_learned_noalloc: " + std::to_string(lanes) +
                                              " lanes exceed the fixed workspace of " +
                                              std::to_string(HWPA_NOALLOC_MAX_LANES) + " lanes");
    unsigned char* base = nullptr;
    int32_t rc = NoAllocScratch(&base);
    if (rc != HWPA_OK) return rc;
    LearnedWs w = CarveLearnedWs(base, lanes);
    hipStream_t s = AsStream(stream);
    rc = DmeEstimateLearned(*cfg, m, w, d_hist, d_stats, d_models, model_fi, est_fi, lanes, d_iters, s);
    if (hipStreamSynchronize(s) != hipSuccess && rc == HWPA_OK) rc = Fail(HWPA_ERR_HIP, "learned EM failed");
    if (rc == HWPA_OK && fallback_count) {
        if (hipMemcpy(fallback_count, w.total + 1, 4, hipMemcpyDeviceToHost) != hipSuccess)
            rc = Fail(HWPA_ERR_HIP, "fallback count copy failed");
    }
    return rc;
}
