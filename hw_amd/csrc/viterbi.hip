// viterbi.hip -- frame labeling: ROI hysteresis prefilter, 13-state subframe
// Viterbi with a 16-frame stitch look-back, traceback and latent update
// (FrameLabelerHost, traceAnalysis/FrameLabelerHost.cpp:53-612; scorer,
// traceAnalysis/SubframeScorer.h:143-318; ROI, traceAnalysis/RoiHost.h:75-248;
// transition matrix, traceAnalysis/SubframeScorer.cpp:35-223).
//
// Mapping: one wave64 per lane, one thread per ZMW (four in small pools, see LabelQuadKernel),
// sequential over frames.
// The ROI is computed first (forward hysteresis, then a backward pass) into a
// 2-bit-per-frame LDS array; the recursion then runs over latent + chunk +
// stitch frames.  The transition matrix has a fixed sparsity (each row: one
// leading column plus one contiguous segment), so the whole predecessor
// choice of a frame packs into one 32-bit word: 4 bits for the baseline row
// and each up row (9 candidates), 1 bit for each full and down row (2
// candidates).  One coalesced 256-byte word row per frame goes to HBM and is
// read back once by the traceback.  Ties pick the later predecessor, as the
// host recursion's `>=` does.

#include "internal.h"

#include <algorithm>
#include <cmath>

namespace hwpa {

struct TransVals {
    float bu[5][5];   // rows B, TU, GU, CU, AU: candidates {B, TU, GU, CU, AU}
    float bd[5];      // the same rows: the one value shared by candidates TD, GD, CD, AD
    float fd[8][2];   // rows T, G, C, A, TD, GD, CD, AD: candidates {full_i, up_i}
};

struct LabLaneState {
    hwpa_lane_model oldModel;
    int16_t labelBoundary[LS];
    uint16_t roiBoundary[LS];
    int16_t latentTrc[LS];
    int16_t prevLat[NL][LS];
};

struct LabelerDev {
    TransVals T;
    float roiUpper, roiLower;
    uint32_t lanes, maxFrames;
    bool quad = false;       // labeled by LabelQuadKernel unless tuned; the buffer holds its words too
    LabLaneState* state = nullptr;
    uint32_t* tb = nullptr;  // [lane][maxFrames + 16 + NS][LS]: predecessor words, then the anchor row;
                             // or (quad) 64-bit words [lane][maxFrames + 16][LS]
};

// Pools of at most this many lanes are labeled by four threads per ZMW (LabelQuadKernel).  It
// issues 1.5 times the instructions of LabelKernel, in waves 2.6 times shorter, so it wins until
// its waves fill the chip's issue slots (512 frames, quad against one thread per ZMW: 16 lanes
// 0.20 against 0.50 ms, 512 lanes 0.32 against 0.52, 1,024 lanes 0.55 against 0.54, 4,096 lanes
// 1.9 against 1.2).  Pools on their own streams, us a chunk with quad and without, for one, three
// and eight pools: 300 lanes 1565, 673, 724 and 1740, 703, 765; 400 lanes 1575, 736, 790 and 1755,
// 728, 793; 512 lanes 1671, 805, 848 and 1846, 762, 828, which one pool gains more than
// three lose.  Pools of one batch count together (six pools of 365 to 2,048 lanes in
// one graph: 7.1 ms a step, 7.3 with the two smallest on four threads).
constexpr uint32_t kQuadLanes = 512;

// nhB = -1/(2 var_B), nhP = -1/(2 var_a): the reference's -0.5f * y * invVar * y
// equals (y * (-0.5f * invVar)) * y bit for bit (scaling by -0.5 is exact here).
struct ScorerZ {
    float bgMean, nhB, bgFixed, x0;
    float ffMean[NA], nhP[NA], ffFixed[NA], logPMean[NA], x1[NA];
    float dimMean, dimNorm, dimScale;
};

// BlockStateSubframeScorer::Setup / SubframeSetup (SubframeScorer.h:151-281)
__device__ void ScorerSetup(ScorerZ& s, const hwpa_lane_model& m, int z)
{
    const float log2pi = 1.8378770664f;
    const float pi = 3.1415926536f;
    const float sqrtHalfPi = hw_sqrtf(0.5f * pi);
    const float bMean = hw_h2f(m.baseline.means[z]);
    const float bVar = hw_h2f(m.baseline.vars[z]);
    const float bSigma = hw_sqrtf(bVar);
    s.x0 = bMean + bSigma * sqrtHalfPi;
    s.nhB = -0.5f * (1.0f / bVar);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        const float aMean = hw_h2f(m.analogs[a].means[z]);
        s.logPMean[a] = hw_cephes_logf(aMean - bMean);
        const float aVar = hw_h2f(m.analogs[a].vars[z]);
        const float aSigma = hw_sqrtf(aVar);
        s.x1[a] = aMean - aSigma * sqrtHalfPi;
        s.nhP[a] = -0.5f * (1.0f / aVar);
    }
    {
        const float aMean = hw_h2f(m.analogs[3].means[z]);
        const float aVar = hw_h2f(m.analogs[3].vars[z]);
        const float eMean = 0.5f * (bMean + aMean);
        float eVar = (1.0f / 6.0f) * (aMean - bMean);
        eVar += bVar + aVar;
        eVar *= 0.5f;
        s.dimMean = eMean;
        s.dimNorm = -0.5f * (log2pi + hw_cephes_logf(eVar));
        s.dimScale = 0.5f / eVar;
    }
    const float normConst = log2pi / 2.0f;
    s.bgFixed = -0.5f * hw_cephes_logf(bVar) - normConst;
    s.bgMean = bMean;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        s.ffFixed[a] = -0.5f * hw_cephes_logf(hw_h2f(m.analogs[a].vars[z])) - normConst;
        s.ffMean[a] = hw_h2f(m.analogs[a].means[z]);
    }
}

// BlockStateSubframeScorer::StateScores for all 13 states (SubframeScorer.h:182-228, 284-305)
__device__ __forceinline__ void Scores(const ScorerZ& s, float d, float* sc)
{
    {
        const float y = d - s.bgMean;
        sc[0] = (y * s.nhB) * y + s.bgFixed;
    }
    float ff[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const float y = d - s.ffMean[i];
        ff[i] = (y * s.nhP[i]) * y + s.ffFixed[i];
        sc[1 + i] = ff[i];
    }
    const bool lowExt = d < s.x0;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const float cap = lowExt ? s.x0 : s.x1[i];
        const float fixedTerm = lowExt ? s.nhB : s.nhP[i];
        const bool ext = lowExt || (d > s.x1[i]);
        const float dc = d - cap;
        float v = (ext ? fixedTerm * (dc * dc) : 0.0f) - s.logPMean[i];
        if (i == NA - 1) {
            const float dm = d - s.dimMean;
            const float fb = s.dimNorm - (dm * dm) * s.dimScale;
            v = (s.x0 <= s.x1[i]) ? v : fb;
        }
        if (d > s.ffMean[i]) v = hw_minf(hw_minf(v, ff[i] - 1.0f), 0.0f);
        sc[5 + i] = v;   // up state
        sc[9 + i] = v;   // down state (same analog, same score)
    }
}

// One Viterbi recursion step (FrameLabelerHost.cpp:213-264): (score + transition) +
// previous log-likelihood per candidate, the later candidate winning ties.  In rows B
// and TU..AU the four down candidates share one transition value, so score + value is
// formed once per row (the same rounded sum the reference forms four times).
// pen = 0 inside the ROI, +inf outside (every state but the baseline is excluded).
__device__ __forceinline__ uint32_t Recur(const TransVals& T, const float* sc, float* ll, float pen)
{
    float acc[NS];
    uint32_t word = 0;
    // The five rows' maximum chains advance together, one candidate at a time, so
    // each compare has independent work behind it before its select.
    float mx[5], sr[5];
    uint32_t code[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        sr[q] = sc[(q == 0) ? 0 : 4 + q];
        mx[q] = (sr[q] + T.bu[q][0]) + ll[0];
        code[q] = 0;
    }
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        if (p == 4) {
#pragma unroll
            for (int q = 0; q < 5; ++q) sr[q] = sr[q] + T.bd[q];
        }
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const float v = (p < 4) ? (sr[q] + T.bu[q][1 + p]) + ll[5 + p] : sr[q] + ll[5 + p];
            const bool c = v >= mx[q];
            mx[q] = c ? v : mx[q];
            code[q] = c ? (uint32_t)(1 + p) : code[q];
        }
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        const int r = (q == 0) ? 0 : 4 + q;
        acc[r] = (r == 0) ? mx[q] : (mx[q] - pen);
        word |= code[q] << (4 * q);
    }
    // full rows 1..4 and down rows 9..12: candidates {full_i, up_i}
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int i = q & 3;
        const int r = (q < 4) ? 1 + i : 9 + i;
        const float s = sc[r];
        const float a = (s + T.fd[q][0]) + ll[1 + i];
        const float b = (s + T.fd[q][1]) + ll[5 + i];
        const bool c = b >= a;
        const float m = c ? b : a;
        acc[r] = m - pen;
        word |= (c ? 1u : 0u) << (20 + q);
    }
#pragma unroll
    for (int r = 0; r < NS; ++r) ll[r] = acc[r];
    return word;
}

__device__ __forceinline__ int Pred(uint32_t w, int state)
{
    if (state == 0 || (state >= 5 && state <= 8)) {
        const int q = (state == 0) ? 0 : state - 4;
        const int code = (int)((w >> (4 * q)) & 15u);
        return code == 0 ? 0 : code + 4;
    }
    const int i = (state <= 4) ? state - 1 : state - 9;
    const int q = (state <= 4) ? i : 4 + i;
    return ((w >> (20 + q)) & 1u) ? 5 + i : 1 + i;
}

// Pred for a state that differs between ZMWs (the traceback): both field lookups and a
// select, no divergent branch.  Shift amounts stay below 32 for every state.
__device__ __forceinline__ int PredSel(uint32_t w, int state)
{
    const uint32_t qb = (state == 0) ? 0u : ((uint32_t)(state - 4) & 7u);
    const int code = (int)((w >> (4u * qb)) & 15u);
    const int pb = code == 0 ? 0 : code + 4;
    const int i = (state <= 4 ? state - 1 : state - 9) & 3;
    const uint32_t q = (uint32_t)((state <= 4) ? i : 4 + i);
    const int pf = ((w >> (20u + q)) & 1u) ? 5 + i : 1 + i;
    const bool bu = state == 0 || (state >= 5 && state <= 8);
    return bu ? pb : pf;
}

// The ROI penalty of the frame whose final ROI bit is bit `pos` of `w`: 0 or +inf.
__device__ __forceinline__ float RoiPen(uint32_t w, uint32_t pos)
{
    const uint32_t m = (uint32_t)__builtin_amdgcn_sbfe((int32_t)w, pos, 1);   // 0 or all ones
    return hw_u2f(~m & 0x7f800000u);
}

// PB = frames per prefetched batch (8 or 16) in the recursion and the traceback.
// MINW = waves per SIMD the register allocation must allow (1: unconstrained).
template <int PB, int MINW>
__global__ __launch_bounds__(64, MINW) void LabelKernel(const int16_t* __restrict__ traces, int frames,
                                                  const hwpa_lane_model* __restrict__ models, LabLaneState* state,
                                                  uint32_t* __restrict__ tbAll, int tbFrames,
                                                  int16_t* __restrict__ labels, int16_t* __restrict__ latentOut,
                                                  float* __restrict__ score, TransVals T, float roiUpper,
                                                  float roiLower)
{
    static_assert(PB % 8 == 0, "recursion batches cover whole 8-frame groups of an ROI word");
    extern __shared__ uint32_t roiWords[];  // [(nroi + 15) / 16][LS], 2 bits per frame
    const int lane = blockIdx.x;
    const int z = threadIdx.x;
    LabLaneState& st = state[lane];
    const hwpa_lane_model& model = models[lane];
    const int16_t* tr = traces + (size_t)lane * frames * LS + z;
    uint32_t* tb = tbAll + (size_t)lane * tbFrames * LS + z;
    const int nroi = frames + HWPA_VITERBI_LOOKBACK + HWPA_ROI_STITCH;
    const int nlab = frames + HWPA_VITERBI_LOOKBACK;
    const int nwords = (nroi + 15) / 16;

    // Latent trace out = the 24 frames preceding this chunk.
    for (int i = 0; i < NL; ++i) latentOut[((size_t)lane * NL + i) * LS + z] = st.prevLat[i][z];

    const float inv1 = 1.0f / hw_sqrtf(hw_h2f(st.oldModel.baseline.vars[z]));
    const float inv2 = 1.0f / hw_sqrtf(hw_h2f(model.baseline.vars[z]));
    // Frame k of the latent ++ chunk sequence (k < NL: the carried latent frames).
    auto rawAt = [&](int k) -> int { return (k < NL) ? (int)st.prevLat[k][z] : (int)tr[(size_t)(k - NL) * LS]; };

    // ROI forward pass (RoiHost.h:137-193) over k < nroi, reading frame k + 2, one
    // 16-frame word at a time with the next word's frames in flight; indices past
    // the sequence re-read its last frame (their values are never used).
    {
        const float kS2 = 1.41421353816986083984375f;   // sqrt(2.0f)
        const float kS3 = 1.73205077648162841796875f;   // sqrt(3.0f)
        const float kR2 = 1.0f / kS2, kR3 = 1.0f / kS3;
        float p0 = (float)st.latentTrc[z] * inv1, p1 = (float)rawAt(0) * inv1, p2 = (float)rawAt(1) * inv1;
        uint32_t prevRoi = st.roiBoundary[z];
        const int limit = nroi + 2;
        auto load16 = [&](int base, int (&dst)[16]) {
#pragma unroll
            for (int u = 0; u < 16; ++u) dst[u] = rawAt(min(base + u, limit - 1));
        };
        auto frame = [&](int k, int raw) -> uint32_t {
            const float nv = (float)raw * ((k + 2 < NL) ? inv1 : inv2);
            const float a2 = p0 + p1;
            const float a3 = a2 + p2;
            const float a4 = a3 + nv;
            float mval = hw_maxf(p1, hw_div_by_const(a2, kS2, kR2));
            mval = hw_maxf(mval, hw_div_by_const(a3, kS3, kR3));
            mval = hw_maxf(mval, a4 * 0.5f);
            const float thresh = (prevRoi & 1u) ? roiLower : roiUpper;
            const uint32_t v = (mval >= thresh ? 1u : 0u) | (mval >= roiLower ? 2u : 0u);
            prevRoi = v;
            p0 = p1;
            p1 = p2;
            p2 = nv;
            return v;
        };
        int cur[16], nxt[16];
        load16(2, cur);
        const int full = nroi / 16;
        for (int wi = 0; wi < full; ++wi) {
            load16(16 * wi + 18, nxt);
            uint32_t word = 0;
#pragma unroll
            for (int u = 0; u < 16; ++u) word |= frame(16 * wi + u, cur[u]) << (2 * u);
            roiWords[wi * LS + z] = word;
#pragma unroll
            for (int u = 0; u < 16; ++u) cur[u] = nxt[u];
        }
        if (full < nwords) {
            uint32_t word = 0;
#pragma unroll
            for (int u = 0; u < 16; ++u)
                if (16 * full + u < nroi) word |= frame(16 * full + u, cur[u]) << (2 * u);
            roiWords[full * LS + z] = word;
        }
    }
    // ROI backward pass (RoiHost.h:195-243), a word at a time: the final ROI bit of
    // each frame into bit 0 of its field (fields past the last frame stay zero).
    {
        uint32_t carry = 0;
        for (int wi = nwords - 1; wi >= 0; --wi)
            roiWords[wi * LS + z] = hw_roi_backward_word(roiWords[wi * LS + z], &carry);
    }

    // Forward recursion over latent, chunk and stitch frames.
    float ll[NS];
    const int lb = st.labelBoundary[z];
#pragma unroll
    for (int s = 0; s < NS; ++s) ll[s] = (lb == s) ? 0.0f : hw_u2f(0xff800000u);
    ScorerZ sc;
    auto step = [&](int f, int raw, uint32_t rw) {
        float s[NS];
        Scores(sc, (float)raw, s);
        tb[(size_t)f * LS] = Recur(T, s, ll, RoiPen(rw, 2u * (uint32_t)(f & 15)));
    };
    // The latent frames are scored with the previous chunk's model, the chunk
    // and stitch frames with the current one.
    ScorerSetup(sc, st.oldModel, z);
    for (int f = 0; f < NL; ++f) step(f, (int)st.prevLat[f][z], roiWords[(f >> 4) * LS + z]);
    // Log-likelihoods at the chunk's last frame, read back once the anchor state is known:
    // kept in the last NS rows of the lane's traceback buffer (13 registers fewer through
    // the stitch frames, no LDS).
    uint32_t* anchorLL = tb + (size_t)(tbFrames - NS) * LS;
    auto storeAnchor = [&]() {
#pragma unroll
        for (int r = 0; r < NS; ++r) anchorLL[(size_t)r * LS] = hw_f2u(ll[r]);
    };
    ScorerSetup(sc, model, z);
    {
        // Chunk frames f in [NL, frames) in batches of PB (f0 a multiple of 8, so each
        // group of 8 frames reads one ROI word) with the next batch in flight, then
        // the remainder; chunk sample j = f - NL.
        const int last = nlab - NL - 1;   // last chunk sample the recursion reads
        auto loadBatch = [&](int j0, int (&dst)[PB]) {
#pragma unroll
            for (int u = 0; u < PB; ++u) dst[u] = (int)tr[(size_t)min(j0 + u, last) * LS];
        };
        const int nb = (frames - NL) / PB;
        int cur[PB], nxt[PB];
        loadBatch(0, cur);
        for (int b = 0; b < nb; ++b) {
            const int f0 = NL + b * PB;
            loadBatch((b + 1) * PB, nxt);
#pragma unroll
            for (int g = 0; g < PB / 8; ++g) {
                const int fg = f0 + 8 * g;
                const uint32_t rw = roiWords[(fg >> 4) * LS + z];
#pragma unroll
                for (int u = 0; u < 8; ++u) step(fg + u, cur[8 * g + u], rw);
            }
#pragma unroll
            for (int u = 0; u < PB; ++u) cur[u] = nxt[u];
        }
        // The remainder of the chunk frames, the anchor, then the stitch frames f in
        // [frames, nlab) (chunk samples frames - NL .. last), one frame at a time with
        // the next sample in flight.
        const int f1 = NL + nb * PB;
        int raw = (int)tr[(size_t)(f1 - NL) * LS];
#pragma unroll 1
        for (int f = f1; f < nlab; ++f) {
            const int nextRaw = (int)tr[(size_t)min(f + 1 - NL, last) * LS];
            if (f == frames) storeAnchor();
            step(f, raw, roiWords[(f >> 4) * LS + z]);
            raw = nextRaw;
        }
    }

    // Normalize and propagate end-state probabilities back 16 frames (FrameLabelerHost.cpp:185-205, 388-417)
    float prob[NS];
    {
        float mx = ll[0];
#pragma unroll
        for (int i = 1; i < NS; ++i) mx = hw_maxf(ll[i], mx);
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            prob[i] = hw_cephes_expf(ll[i] - mx);
            sum += prob[i];
        }
        const float inv = 1 / sum;
#pragma unroll
        for (int i = 0; i < NS; ++i) prob[i] *= inv;
    }
    for (int i = nlab - 1; i > frames - 1; --i) {
        const uint32_t w = tb[(size_t)i * LS];
        float np[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) np[s] = 0.0f;
#pragma unroll
        for (int from = 0; from < NS; ++from) {
            const int ps = Pred(w, from);
#pragma unroll
            for (int to = 0; to < NS; ++to) np[to] += (to == ps) ? prob[from] : 0.0f;
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) prob[s] = np[s];
    }
    float maxProb = prob[0];
    int anchorState = 0;
#pragma unroll
    for (int i = 1; i < NS; ++i) {
        const bool cond = maxProb > prob[i];
        maxProb = cond ? maxProb : prob[i];
        anchorState = cond ? anchorState : i;
    }
    const float sv = hw_u2f(anchorLL[(size_t)anchorState * LS]);
    score[(size_t)lane * LS + z] = sv;

    // Traceback from the anchor, PB predecessor words per batch with the next batch in
    // flight, then the remainder.
    int16_t* lo = labels + (size_t)lane * frames * LS + z;
    int stt = anchorState;
    {
        auto loadTb = [&](int top, uint32_t (&dst)[PB]) {
#pragma unroll
            for (int u = 0; u < PB; ++u) dst[u] = tb[(size_t)max(top - u, 0) * LS];
        };
        const int nb = frames / PB;
        uint32_t cur[PB], nxt[PB];
        loadTb(frames - 1, cur);
        for (int b = 0; b < nb; ++b) {
            const int top = frames - 1 - b * PB;
            loadTb(top - PB, nxt);
#pragma unroll
            for (int u = 0; u < PB; ++u) {
                lo[(size_t)(top - u) * LS] = (int16_t)stt;
                stt = PredSel(cur[u], stt);
            }
#pragma unroll
            for (int u = 0; u < PB; ++u) cur[u] = nxt[u];
        }
#pragma unroll 1
        for (int f = frames - 1 - nb * PB; f >= 0; --f) {
            lo[(size_t)f * LS] = (int16_t)stt;
            stt = PredSel(tb[(size_t)f * LS], stt);
        }
    }

    // Latent update
    const int anchor = frames - NL;
    const int fl = frames - 1;
    st.roiBoundary[z] = (uint16_t)((roiWords[(fl >> 4) * LS + z] >> (2 * (fl & 15))) & 1u);
    st.labelBoundary[z] = (int16_t)anchorState;
    st.latentTrc[z] = tr[(size_t)(anchor - 1) * LS];
    for (int i = 0; i < NL; ++i) st.prevLat[i][z] = tr[(size_t)(anchor + i) * LS];
    // Model copy (each thread copies its ZMW column)
    st.oldModel.baseline.means[z] = model.baseline.means[z];
    st.oldModel.baseline.vars[z] = model.baseline.vars[z];
    st.oldModel.baseline.weights[z] = model.baseline.weights[z];
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        st.oldModel.analogs[a].means[z] = model.analogs[a].means[z];
        st.oldModel.analogs[a].vars[z] = model.analogs[a].vars[z];
        st.oldModel.analogs[a].weights[z] = model.analogs[a].weights[z];
    }
    st.oldModel.confidence[z] = model.confidence[z];
}

// ---- four threads per ZMW -----------------------------------------------------
// For pools that leave the chip partly idle: a quad of lanes carries one ZMW, thread a of it the
// states of analog a (full_a, up_a, down_a; the baseline state is kept by all four), so a wave
// holds 16 ZMWs and a frame costs it 168 instructions instead of 440.  Values cross the quad by DPP.  A frame's predecessor choices are one 64-bit word per
// ZMW, 16 bits from each thread: the nibbles of full_a, up_a, down_a and the baseline, at the
// state's own nibble index (4a, 4a + 1, 4a + 2; 3 for the baseline), each holding the
// predecessor's index, so a traceback step is one shift of that word.
// Every value is formed as LabelKernel forms it, so both give the same bits.

template <int CTRL>
__device__ __forceinline__ uint32_t QuadU(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float QuadF(float v) { return hw_u2f(QuadU<CTRL>(hw_f2u(v))); }
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;
// Value of quad thread P.
template <int P>
__device__ __forceinline__ float QuadAt(float v) { return QuadF<P * 0x55>(v); }
__device__ __forceinline__ float QuadAt(float v, int p)
{
    return p == 0 ? QuadAt<0>(v) : p == 1 ? QuadAt<1>(v) : p == 2 ? QuadAt<2>(v) : QuadAt<3>(v);
}
__device__ __forceinline__ uint32_t QuadAtU(uint32_t v, int p)
{
    return p == 0 ? QuadU<0x00>(v) : p == 1 ? QuadU<0x55>(v) : p == 2 ? QuadU<0xAA>(v) : QuadU<0xFF>(v);
}
__device__ __forceinline__ uint32_t QuadOr(uint32_t v)
{
    v |= QuadU<kQuadXor1>(v);
    return v | QuadU<kQuadXor2>(v);
}
__device__ __forceinline__ uint32_t QuadMaxU(uint32_t v)
{
    v = max(v, QuadU<kQuadXor1>(v));
    return max(v, QuadU<kQuadXor2>(v));
}

constexpr uint32_t kNibB = 3;   // nibble index of the baseline state
// State number of a nibble index: full_a 1 + a, up_a 5 + a, down_a 9 + a, the baseline 0.
__device__ __forceinline__ int NibState(uint32_t n)
{
    const int k = (int)(n & 3u);
    return k == 3 ? 0 : 1 + (int)(n >> 2) + 4 * k;
}
__device__ __forceinline__ uint32_t StateNib(int s) { return s == 0 ? kNibB : 4u * (uint32_t)((s - 1) & 3) + (uint32_t)((s - 1) >> 2); }

struct ScorerQ {   // ScorerZ's values for the baseline and one analog
    float bgMean, nhB, bgFixed, x0;
    float ffMean, nhP, ffFixed, logPMean, x1;
    float dimMean, dimNorm, dimScale;
    bool dim;      // the last analog's fallback score applies (x0 > x1)
};

__device__ void ScorerSetupQuad(ScorerQ& q, const hwpa_lane_model& m, int z, int a)
{
    const float log2pi = 1.8378770664f;
    const float pi = 3.1415926536f;
    const float sqrtHalfPi = hw_sqrtf(0.5f * pi);
    const float bMean = hw_h2f(m.baseline.means[z]);
    const float bVar = hw_h2f(m.baseline.vars[z]);
    const float bSigma = hw_sqrtf(bVar);
    const float normConst = log2pi / 2.0f;
    q.x0 = bMean + bSigma * sqrtHalfPi;
    q.nhB = -0.5f * (1.0f / bVar);
    q.bgFixed = -0.5f * hw_cephes_logf(bVar) - normConst;
    q.bgMean = bMean;
    const float aMean = hw_h2f(m.analogs[a].means[z]);
    const float aVar = hw_h2f(m.analogs[a].vars[z]);
    const float aSigma = hw_sqrtf(aVar);
    q.logPMean = hw_cephes_logf(aMean - bMean);
    q.x1 = aMean - aSigma * sqrtHalfPi;
    q.nhP = -0.5f * (1.0f / aVar);
    q.ffFixed = -0.5f * hw_cephes_logf(aVar) - normConst;
    q.ffMean = aMean;
    // (the fallback's values; used by the last analog only)
    const float eMean = 0.5f * (bMean + aMean);
    float eVar = (1.0f / 6.0f) * (aMean - bMean);
    eVar += bVar + aVar;
    eVar *= 0.5f;
    q.dimMean = eMean;
    q.dimNorm = -0.5f * (log2pi + hw_cephes_logf(eVar));
    q.dimScale = 0.5f / eVar;
    q.dim = a == NA - 1 && !(q.x0 <= q.x1);
}

struct TransQ {    // a thread's part of TransVals
    float b0, bu, bd;          // row B: candidates B, up_a, and the down states
    float u0, uu[NA], ud;      // row up_a: candidates B, the up states, the down states
    float f0, f1, d0, d1;      // rows full_a and down_a: candidates full_a, up_a
};

__global__ __launch_bounds__(256) void LabelQuadKernel(const int16_t* __restrict__ traces, int frames,
                                                       const hwpa_lane_model* __restrict__ models,
                                                       LabLaneState* state, uint16_t* __restrict__ tbAll, int tbFrames,
                                                       int16_t* __restrict__ labels, int16_t* __restrict__ latentOut,
                                                       float* __restrict__ score, TransVals T, float roiUpper,
                                                       float roiLower)
{
    extern __shared__ uint32_t roiWords[];   // [(nroi + 15) / 16][LS], 2 bits per frame; a wave uses its own columns
    const int lane = blockIdx.x;
    const int a = threadIdx.x & 3;
    const int z = threadIdx.x >> 2;
    LabLaneState& st = state[lane];
    const hwpa_lane_model& model = models[lane];
    const int16_t* tr = traces + (size_t)lane * frames * LS + z;
    uint16_t* tb = tbAll + ((size_t)lane * tbFrames * LS + z) * 4;   // [frame][ZMW][4]
    const int nroi = frames + HWPA_VITERBI_LOOKBACK + HWPA_ROI_STITCH;
    const int nlab = frames + HWPA_VITERBI_LOOKBACK;
    const int nwords = (nroi + 15) / 16;

#pragma unroll
    for (int i = 0; i < NL; i += 4) latentOut[((size_t)lane * NL + i + a) * LS + z] = st.prevLat[i + a][z];

    const float inv1 = 1.0f / hw_sqrtf(hw_h2f(st.oldModel.baseline.vars[z]));
    const float inv2 = 1.0f / hw_sqrtf(hw_h2f(model.baseline.vars[z]));
    // Frame k of the latent ++ chunk sequence, from a selected address (no branch).
    const int seq = NL + frames;
    auto rawAt = [&](int k) -> int {
        const int16_t* p = (k < NL) ? &st.prevLat[k][z] : tr + (size_t)(k - NL) * LS;
        return (int)*p;
    };

    // ROI forward pass: thread a compares frames 4a .. 4a + 3 of each 16-frame word with both
    // thresholds (the sums of a frame depend on the frames around it only); the hysteresis
    // then runs over the word's bits: r_k = r_{k-1} ? (m_k >= lower) : (m_k >= upper).
    {
        const float kS2 = 1.41421353816986083984375f;   // sqrt(2.0f)
        const float kS3 = 1.73205077648162841796875f;   // sqrt(3.0f)
        const float kR2 = 1.0f / kS2, kR3 = 1.0f / kS3;
        uint32_t carry = st.roiBoundary[z] & 1u;
        const int firstRaw = (int)st.latentTrc[z];
        // Frames 16 w + 4 a - 1 .. + 5 (frame -1 is the one before the latent frames; frames
        // past the sequence re-read its last one and are not used).
        auto load = [&](int w, int (&dst)[7]) {
#pragma unroll
            for (int u = 0; u < 7; ++u) dst[u] = rawAt(min(max(16 * w + 4 * a - 1 + u, 0), seq - 1));
        };
        int cur[7], nxt[7];
        load(0, cur);
        for (int w = 0; w < nwords; ++w) {
            load(w + 1, nxt);
            float n[7];
#pragma unroll
            for (int u = 0; u < 7; ++u) {
                const int k = 16 * w + 4 * a - 1 + u;
                n[u] = (float)((k < 0) ? firstRaw : cur[u]) * ((k < NL) ? inv1 : inv2);
            }
            uint32_t up = 0, low = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float a2 = n[u] + n[u + 1];
                const float a3 = a2 + n[u + 2];
                const float a4 = a3 + n[u + 3];
                float mval = hw_maxf(n[u + 1], hw_div_by_const(a2, kS2, kR2));
                mval = hw_maxf(mval, hw_div_by_const(a3, kS3, kR3));
                mval = hw_maxf(mval, a4 * 0.5f);
                const bool in = 16 * w + 4 * a + u < nroi;
                up |= (in && mval >= roiUpper) ? 1u << (2 * u) : 0u;
                low |= (in && mval >= roiLower) ? 1u << (2 * u) : 0u;
            }
            const uint32_t U = QuadOr(up << (8 * a)), L = QuadOr(low << (8 * a));
            uint32_t R = 0;
            if (roiUpper >= roiLower) {
                // U implies L: r_k = u_k | (l_k & r_{k-1}) is the carry chain of one addition.
                const uint32_t g = U << 1, pr = L << 1;
                const uint32_t x = g | pr | 0x55555555u;
                const uint32_t cin = (x + g + carry) ^ x ^ g;
                R = (g | (pr & cin)) >> 1;
                carry = (R >> 30) & 1u;
            } else {
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    carry = ((carry ? L : U) >> (2 * k)) & 1u;
                    R |= carry << (2 * k);
                }
            }
            if (a == 0) roiWords[w * LS + z] = R | (L << 1);
#pragma unroll
            for (int u = 0; u < 7; ++u) cur[u] = nxt[u];
        }
    }
    // ROI backward pass, a word at a time (all four threads form the same word).  The words pass
    // between lanes of one wave only, whose LDS and memory accesses stay in order: the fences keep
    // the compiler from moving them.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    {
        uint32_t carry = 0;
        for (int wi = nwords - 1; wi >= 0; --wi) {
            const uint32_t v = hw_roi_backward_word(roiWords[wi * LS + z], &carry);
            if (a == 0) roiWords[wi * LS + z] = v;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    TransQ t;
    t.b0 = T.bu[0][0];
    t.bd = T.bd[0];
    t.bu = a == 0 ? T.bu[0][1] : a == 1 ? T.bu[0][2] : a == 2 ? T.bu[0][3] : T.bu[0][4];
    {
        auto pick = [&](float v0, float v1, float v2, float v3) { return a == 0 ? v0 : a == 1 ? v1 : a == 2 ? v2 : v3; };
        t.u0 = pick(T.bu[1][0], T.bu[2][0], T.bu[3][0], T.bu[4][0]);
#pragma unroll
        for (int p = 0; p < NA; ++p) t.uu[p] = pick(T.bu[1][1 + p], T.bu[2][1 + p], T.bu[3][1 + p], T.bu[4][1 + p]);
        t.ud = pick(T.bd[1], T.bd[2], T.bd[3], T.bd[4]);
        t.f0 = pick(T.fd[0][0], T.fd[1][0], T.fd[2][0], T.fd[3][0]);
        t.f1 = pick(T.fd[0][1], T.fd[1][1], T.fd[2][1], T.fd[3][1]);
        t.d0 = pick(T.fd[4][0], T.fd[5][0], T.fd[6][0], T.fd[7][0]);
        t.d1 = pick(T.fd[4][1], T.fd[5][1], T.fd[6][1], T.fd[7][1]);
    }
    const uint32_t nibF = 4u * (uint32_t)a, nibU = nibF + 1u, nibD = nibF + 2u;

    float lB, lF, lU, lD;
    {
        const float ninf = hw_u2f(0xff800000u);
        const int lb = st.labelBoundary[z];
        lB = lb == 0 ? 0.0f : ninf;
        lF = lb == 1 + a ? 0.0f : ninf;
        lU = lb == 5 + a ? 0.0f : ninf;
        lD = lb == 9 + a ? 0.0f : ninf;
    }
    ScorerQ sc;
    // One frame: Scores and Recur of LabelKernel.
    auto step = [&](int f, float d, uint32_t rw) {
        const float pen = RoiPen(rw, 2u * (uint32_t)(f & 15));
        float y = d - sc.bgMean;
        const float sB = (y * sc.nhB) * y + sc.bgFixed;
        y = d - sc.ffMean;
        const float sF = (y * sc.nhP) * y + sc.ffFixed;
        const bool lowExt = d < sc.x0;
        const float cap = lowExt ? sc.x0 : sc.x1;
        const float fixedTerm = lowExt ? sc.nhB : sc.nhP;
        const bool ext = lowExt || (d > sc.x1);
        const float dc = d - cap;
        float s = (ext ? fixedTerm * (dc * dc) : 0.0f) - sc.logPMean;
        {
            const float dm = d - sc.dimMean;
            const float fb = sc.dimNorm - (dm * dm) * sc.dimScale;
            s = sc.dim ? fb : s;
        }
        if (d > sc.ffMean) s = hw_minf(hw_minf(s, sF - 1.0f), 0.0f);

        // Row B.  The running maximum over {B, up 0-3, down 0-3} with later candidates winning
        // ties, a NaN candidate never winning and a NaN first one never replaced, equals: the
        // (IEEE) maximum of the eight, the last of them that reaches it, taken if >= B's.
        const float cB = (sB + t.b0) + lB;
        const float cU = (sB + t.bu) + lU;
        const float cD = (sB + t.bd) + lD;
        float m8 = __builtin_fmaxf(cU, cD);
        m8 = __builtin_fmaxf(m8, QuadF<kQuadXor1>(m8));
        m8 = __builtin_fmaxf(m8, QuadF<kQuadXor2>(m8));
        uint32_t code = (cU == m8) ? 1u + (uint32_t)a : 0u;
        code = (cD == m8) ? 5u + (uint32_t)a : code;
        code = QuadMaxU(code);
        const bool takeB = m8 >= cB;
        const float nB = takeB ? m8 : cB;
        // candidate code -> nibble index: 0 the baseline, 1 + p up_p, 5 + p down_p
        const uint32_t kB = takeB ? (4u * code - (code > 4u ? 18u : 3u)) : kNibB;

        // Row up_a, candidate by candidate.
        float mx = (s + t.u0) + lB;
        uint32_t kU = kNibB;
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            const float v = (s + t.uu[p]) + QuadAt(lU, p);
            const bool c = v >= mx;
            mx = c ? v : mx;
            kU = c ? 4u * (uint32_t)p + 1u : kU;
        }
        const float sd = s + t.ud;
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            const float v = sd + QuadAt(lD, p);
            const bool c = v >= mx;
            mx = c ? v : mx;
            kU = c ? 4u * (uint32_t)p + 2u : kU;
        }
        // Rows full_a and down_a: candidates {full_a, up_a}.
        const float fa = (sF + t.f0) + lF, fb = (sF + t.f1) + lU;
        const bool cF = fb >= fa;
        const float da = (s + t.d0) + lF, db = (s + t.d1) + lU;
        const bool cDn = db >= da;
        lF = (cF ? fb : fa) - pen;
        lD = (cDn ? db : da) - pen;
        lU = mx - pen;
        lB = nB;
        uint32_t w = cF ? nibU : nibF;
        w |= kU << 4;
        w |= (cDn ? nibU : nibF) << 8;
        w |= kB << 12;
        tb[(size_t)f * LS * 4 + a] = (uint16_t)w;
    };
    // Frames [f0, f1) of the sequence, four at a time when f0 is a multiple of 4 (so the four
    // share an ROI word) with the next sixteen samples in flight: thread a holds frame 4 g + a of
    // each group.
    auto run = [&](int f0, int f1) {
        const bool whole = (f0 & 3) == 0;
        auto sample = [&](int g) { return rawAt(min(f0 + 4 * g + a, seq - 1)); };
        int nx[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) nx[q] = sample(q);
        int g = 0;
        for (; whole && f0 + 16 * (g + 1) <= f1; ++g) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float mine = (float)nx[q];
                nx[q] = sample(4 * (g + 1) + q);
                const int fq = f0 + 16 * g + 4 * q;
                const uint32_t rw = roiWords[(fq >> 4) * LS + z];
#pragma unroll
                for (int u = 0; u < 4; ++u) step(fq + u, QuadAt(mine, u), rw);
            }
        }
        // The remainder, frame by frame (its samples are read by all four threads).
        int f = f0 + 16 * g;
        int raw = rawAt(min(f, seq - 1));
#pragma unroll 1
        for (; f < f1; ++f) {
            const int next = rawAt(min(f + 1, seq - 1));
            step(f, (float)raw, roiWords[(f >> 4) * LS + z]);
            raw = next;
        }
    };
    // The latent frames are scored with the previous chunk's model, the chunk and stitch frames
    // with the current one; the log-likelihoods at the chunk's last frame are kept.
    ScorerSetupQuad(sc, st.oldModel, z, a);
    run(0, NL);
    ScorerSetupQuad(sc, model, z, a);
    run(NL, frames);
    const float aB = lB, aF = lF, aU = lU, aD = lD;
    run(frames, nlab);

    // Normalise and propagate the end-state probabilities back over the stitch frames.
    float pB, pF, pU, pD;
    {
        float all[NS];
        all[0] = lB;
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            all[1 + p] = QuadAt(lF, p);
            all[5 + p] = QuadAt(lU, p);
            all[9 + p] = QuadAt(lD, p);
        }
        float mx = all[0];
#pragma unroll
        for (int i = 1; i < NS; ++i) mx = hw_maxf(all[i], mx);
        pB = hw_cephes_expf(lB - mx);
        pF = hw_cephes_expf(lF - mx);
        pU = hw_cephes_expf(lU - mx);
        pD = hw_cephes_expf(lD - mx);
        float sum = 0.0f;
        sum += pB;
#pragma unroll
        for (int p = 0; p < NA; ++p) sum += QuadAt(pF, p);
#pragma unroll
        for (int p = 0; p < NA; ++p) sum += QuadAt(pU, p);
#pragma unroll
        for (int p = 0; p < NA; ++p) sum += QuadAt(pD, p);
        const float inv = 1 / sum;
        pB *= inv;
        pF *= inv;
        pU *= inv;
        pD *= inv;
    }
#pragma unroll 1
    for (int i = nlab - 1; i > frames - 1; --i) {
        // What each state passes to its predecessor, added in state order (a state's own sum
        // gets +0 from the others, which leaves it as it is).
        const uint32_t w = tb[(size_t)i * LS * 4 + a];
        const uint32_t kB = (w >> 12) & 15u, kU = (w >> 4) & 15u, kF = w & 15u, kD = (w >> 8) & 15u;
        float qU[NA];
        uint32_t jU[NA];
#pragma unroll
        for (int p = 0; p < NA; ++p) {
            qU[p] = QuadAt(pU, p);
            jU[p] = QuadAtU(kU, p);
        }
        auto into = [&](uint32_t n, bool own) {
            float v = 0.0f;
            v += (kB == n) ? pB : 0.0f;
            if (own) v += (kF == n) ? pF : 0.0f;
#pragma unroll
            for (int p = 0; p < NA; ++p) v += (jU[p] == n) ? qU[p] : 0.0f;
            if (own) v += (kD == n) ? pD : 0.0f;
            return v;
        };
        const float nB = into(kNibB, false), nF = into(nibF, true), nU = into(nibU, true), nD = into(nibD, false);
        pB = nB;
        pF = nF;
        pU = nU;
        pD = nD;
    }
    float maxProb = pB, sv = aB;
    int anchorState = 0;
    auto consider = [&](float p, float ll, int i) {
        const bool cond = maxProb > p;
        maxProb = cond ? maxProb : p;
        sv = cond ? sv : ll;
        anchorState = cond ? anchorState : i;
    };
#pragma unroll
    for (int p = 0; p < NA; ++p) consider(QuadAt(pF, p), QuadAt(aF, p), 1 + p);
#pragma unroll
    for (int p = 0; p < NA; ++p) consider(QuadAt(pU, p), QuadAt(aU, p), 5 + p);
#pragma unroll
    for (int p = 0; p < NA; ++p) consider(QuadAt(pD, p), QuadAt(aD, p), 9 + p);
    if (a == 0) score[(size_t)lane * LS + z] = sv;

    // Traceback: thread a reads the whole 64-bit words of frames top - a - 4 q and writes their
    // labels; every thread follows the path.
    {
        int16_t* lo = labels + (size_t)lane * frames * LS + z;
        typedef uint32_t Word64 __attribute__((ext_vector_type(2), may_alias));
        const Word64* tw = reinterpret_cast<const Word64*>(tb);   // [frame][ZMW]
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        uint32_t n = StateNib(anchorState);
        auto word = [&](int top) { return tw[(size_t)max(top - a, 0) * LS]; };
        Word64 nx[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) nx[q] = word(frames - 1 - 4 * q);
        for (int top = frames - 1; top >= 0; top -= 16) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const Word64 w = nx[q];
                nx[q] = word(top - 16 - 4 * q);
                uint32_t mine = 0;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    mine = (a == u) ? n : mine;
                    const uint64_t v = (uint64_t)QuadAtU(w.x, u) | ((uint64_t)QuadAtU(w.y, u) << 32);
                    n = (uint32_t)(v >> (4u * n)) & 15u;
                }
                const int f = top - 4 * q - a;
                if (f >= 0) lo[(size_t)f * LS] = (int16_t)NibState(mine);
            }
        }
    }

    // Latent update
    const int anchor = frames - NL;
    const int fl = frames - 1;
    int16_t lat[NL / 4];
#pragma unroll
    for (int i = 0; i < NL / 4; ++i) lat[i] = tr[(size_t)(anchor + 4 * i + a) * LS];
#pragma unroll
    for (int i = 0; i < NL / 4; ++i) st.prevLat[4 * i + a][z] = lat[i];
    if (a == 0) {
        st.roiBoundary[z] = (uint16_t)((roiWords[(fl >> 4) * LS + z] >> (2 * (fl & 15))) & 1u);
        st.labelBoundary[z] = (int16_t)anchorState;
        st.latentTrc[z] = tr[(size_t)(anchor - 1) * LS];
        st.oldModel.baseline.means[z] = model.baseline.means[z];
        st.oldModel.baseline.vars[z] = model.baseline.vars[z];
        st.oldModel.baseline.weights[z] = model.baseline.weights[z];
        st.oldModel.confidence[z] = model.confidence[z];
    }
    st.oldModel.analogs[a].means[z] = model.analogs[a].means[z];
    st.oldModel.analogs[a].vars[z] = model.analogs[a].vars[z];
    st.oldModel.analogs[a].weights[z] = model.analogs[a].weights[z];
}

__global__ __launch_bounds__(64) void LabelInitKernel(LabLaneState* state)
{
    LabLaneState& st = state[blockIdx.x];
    const int z = threadIdx.x;
    // LatentViterbi ctor (FrameLabelerHost.cpp:58-81)
    st.oldModel.baseline.means[z] = hw_f2h(0.0f);
    st.oldModel.baseline.vars[z] = hw_f2h(50.0f);
    st.oldModel.baseline.weights[z] = 0;
    for (int a = 0; a < NA; ++a) {
        st.oldModel.analogs[a].means[z] = hw_f2h(1000.0f);
        st.oldModel.analogs[a].vars[z] = hw_f2h(10.0f);
        st.oldModel.analogs[a].weights[z] = 0;
    }
    st.oldModel.confidence[z] = 0;
    st.labelBoundary[z] = 0;
    st.roiBoundary[z] = 0;
    st.latentTrc[z] = 0;
    for (int i = 0; i < NL; ++i) st.prevLat[i][z] = 0;
}

// TransitionMatrix<float> ctor (SubframeScorer.cpp:35-223), computed on the host.
void BuildTransition(const hwpa_config& cfg, hwpa_transition& T)
{
    hwpa_analog analogs[NA];
    for (int i = 0; i < NA; ++i) analogs[i] = cfg.movie.analogs[i];
    float data[NS][NS];
    for (int i = 0; i < NS; ++i)
        for (int j = 0; j < NS; ++j) data[i][j] = 0.0f;
    for (int i = 0; i < NA; ++i) {
        const float delta = 0.01f;
        // The first check tests the IPD ratio but adjusts the pulse-width ratio,
        // as the reference does.
        if (std::abs(analogs[i].ipd2_slow_step_ratio - 1.0f) < delta)
            analogs[i].pw2_slow_step_ratio = (analogs[i].pw2_slow_step_ratio < 1.0f) ? 1.0f - delta : 1.0f + delta;
        if (std::abs(analogs[i].ipd2_slow_step_ratio - 1.0f) < delta)
            analogs[i].ipd2_slow_step_ratio = (analogs[i].ipd2_slow_step_ratio < 1.0f) ? 1.0f - delta : 1.0f + delta;
    }
    float meanIpd = 0.0f;
    for (int i = 0; i < NA; ++i) meanIpd += analogs[i].inter_pulse_distance;
    meanIpd = meanIpd / NA;
    const double frameRate = cfg.movie.frame_rate;
    // Probabilities of 1-, 2- and 3-frame events for a two-step kinetic model
    // (double precision, as in the host computation).
    auto lenProbs = [&](float widthSeconds, float ratio, float* ret) {
        const double widthFrames = frameRate * widthSeconds;
        ratio = std::max(ratio, 1e-6f);
        const double k1 = (1.0f + ratio) / widthFrames;
        const double k2 = (1.0f + 1.0f / ratio) / widthFrames;
        const double dk = k1 - k2;
        const double c1 = 1.0f - std::exp(-k1);
        const double c2 = 1.0f - std::exp(-k2);
        ret[0] = (float)(1 - k1 * c2 / k2 / dk + k2 * c1 / k1 / dk);
        ret[1] = (float)(k1 * (c2 * c2) / k2 / dk - k2 * (c1 * c1) / k1 / dk);
        ret[2] = (float)(k1 * (c2 * c2) * (1 - c2) / k2 / dk - k2 * (c1 * c1) * (1 - c1) / k1 / dk);
    };
    float ipdLen[NA][3];
    for (int i = 0; i < NA; ++i) lenProbs(analogs[i].inter_pulse_distance, analogs[i].ipd2_slow_step_ratio, ipdLen[i]);
    float alpha[NA];
    for (int i = 0; i < NA; ++i) alpha[i] = cfg.viterbi_alpha * 0.25f * (ipdLen[i][0] + ipdLen[i][1]);
    float alphaSum = 0.0f;
    for (int i = 0; i < NA; ++i) alphaSum += alpha[i];
    float meanLen[3];
    lenProbs(meanIpd, 0.0f, meanLen);
    const float meanIpd3m = 1 - meanLen[0] - meanLen[1];
    const float pulseStartProb = meanLen[2] / meanIpd3m;
    data[0][0] = 1.0f - pulseStartProb;
    for (int i = 0; i < NA; ++i) {
        const int full = i + 1, up = i + 1 + NA, down = i + 1 + 2 * NA;
        float al[3];
        lenProbs(analogs[i].pulse_width, analogs[i].pw2_slow_step_ratio, al);
        const float gamma = cfg.viterbi_gamma * al[0] / (1 + alphaSum);
        const float beta = cfg.viterbi_beta * al[1];
        data[up][0] = 0.25f * pulseStartProb;
        data[0][up] = gamma;
        data[down][up] = beta;
        data[full][up] = 1 - gamma - gamma * alphaSum - beta;
        const float prob3ms = 1.0f - al[0] - al[1];
        data[down][full] = al[2] / prob3ms;
        data[full][full] = 1.0f - data[down][full];
        data[0][down] = 1 - alphaSum;
        for (int j = 0; j < NA; ++j) {
            const int upPrime = j + 1 + NA;
            data[upPrime][down] = alpha[j];
            data[upPrime][up] = gamma * alpha[j];
        }
    }
    for (int r = 0; r < NS; ++r) {
        if (r == 0 || (r >= 5 && r <= 8)) {
            T.first_col[r] = 0;
            T.seg_first[r] = 5;
            T.seg_last[r] = 13;
        } else {
            const int a = (r <= 4) ? r - 1 : r - 9;
            T.first_col[r] = a + 1;
            T.seg_first[r] = a + 5;
            T.seg_last[r] = a + 6;
        }
    }
    // Entries with probability <= 0 keep the storage's initial 0 (SubframeScorer.cpp:213-220).
    for (int i = 0; i < NS; ++i)
        for (int j = 0; j < NS; ++j) T.logp[i][j] = (data[i][j] > 0.0f) ? std::log(data[i][j]) : 0.0f;
}

// Packs the transition matrix into the kernel's candidate order.  Fails when the
// four down candidates of a row B / TU..AU do not share one value (the matrix the
// reference builds always has that form: SubframeScorer.cpp:173-200).
static bool PackTransition(const hwpa_transition& T, TransVals& v)
{
    v = TransVals{};
    const int buRows[5] = {0, 5, 6, 7, 8};
    for (int q = 0; q < 5; ++q) {
        const int r = buRows[q];
        v.bu[q][0] = T.logp[r][0];
        for (int p = 0; p < 4; ++p) v.bu[q][1 + p] = T.logp[r][5 + p];
        v.bd[q] = T.logp[r][9];
        for (int p = 10; p < 13; ++p)
            if (hw_f2u(T.logp[r][p]) != hw_f2u(v.bd[q])) return false;
    }
    for (int q = 0; q < 8; ++q) {
        const int i = q & 3;
        const int r = (q < 4) ? 1 + i : 9 + i;
        v.fd[q][0] = T.logp[r][1 + i];
        v.fd[q][1] = T.logp[r][5 + i];
    }
    return true;
}

int32_t LabelerCreate(const hwpa_config& cfg, uint32_t lanes, uint32_t max_frames, LabelerDev** out, uint64_t sideBySide)
{
    if (max_frames < (uint32_t)NL) return Fail(HWPA_ERR_INVALID_ARG, "labeler: max_frames must be >= 24");
    hwpa_transition T;
    BuildTransition(cfg, T);
    TransVals packed;
    if (!PackTransition(T, packed))
        return Fail(HWPA_ERR_INVALID_ARG, "labeler: transition rows do not share their down-state values");
    auto* l = new LabelerDev;
    l->T = packed;
    l->roiUpper = cfg.roi_upper_threshold;
    l->roiLower = cfg.roi_lower_threshold;
    l->lanes = lanes;
    l->maxFrames = max_frames;
    int32_t rc = DeviceAlloc((void**)&l->state, sizeof(LabLaneState) * lanes, "labeler state");
    l->quad = std::max<uint64_t>(lanes, sideBySide) <= kQuadLanes;
    if (rc == HWPA_OK) {
        const size_t rows = max_frames + HWPA_VITERBI_LOOKBACK;
        const size_t words = l->quad ? std::max<size_t>(rows + NS, 2 * rows) : rows + NS;
        rc = DeviceAlloc((void**)&l->tb, (size_t)lanes * words * LS * sizeof(uint32_t), "labeler traceback");
    }
    if (rc == HWPA_OK) {
        hipLaunchKernelGGL(LabelInitKernel, dim3(lanes), dim3(LS), 0, nullptr, l->state);
        rc = CheckLaunch("LabelInitKernel");
    }
    if (rc == HWPA_OK && hipDeviceSynchronize() != hipSuccess) rc = Fail(HWPA_ERR_HIP, "labeler init failed");
    if (rc != HWPA_OK) {
        LabelerDestroy(l);
        return rc;
    }
    *out = l;
    return HWPA_OK;
}

void LabelerDestroy(LabelerDev* l)
{
    if (!l) return;
    DeviceFree(l->state);
    DeviceFree(l->tb);
    delete l;
}

// Four threads per ZMW for small pools (kQuadLanes), <16, 4> for 4,096 lanes and more of chunks up to
// 512 frames, else <8, 1>.  Four waves per SIMD pay once there are as many, 4,096 lanes (512 frames,
// <8, 1> and <16, 4>: 1,024 lanes 0.49 and 0.53 ms, 2,048 0.66 and 0.68, 3,072 0.91 and 0.94, 4,096
// 1.20 and 1.17, 8,192 2.23 and 2.18, 16,384 4.27 and 4.22; 256 frames: 3,072 0.50 and 0.51, 4,096
// 0.66 and 0.64, 8,192 1.21 and 1.17), and as long as their ROI words fit a CU's LDS, up to 618 frames
// (4,096 lanes: 576 frames 1.34 and 1.31, 640 frames 1.47 and 1.78, 1024 frames 2.96 and 3.47; 8,192
// lanes: 576 frames 2.48 and 2.47, 640 frames 2.74 and 3.12): the line lies at the usual length below.
int32_t LabelerDefault(const LabelerDev* l, uint32_t frames)
{
    if (l->quad) return 0;
    return (l->lanes >= 4096 && frames <= 512) ? 3 : 1;
}

int32_t LabelerRun(LabelerDev* l, const int16_t* traces, uint32_t frames, const hwpa_lane_model* models,
                   int16_t* labels, int16_t* latent_out, float* score, hipStream_t s)
{
    if (!l || !traces || !models || !labels || !latent_out || !score)
        return Fail(HWPA_ERR_INVALID_ARG, "labeler_run: null argument");
    if (frames <= (uint32_t)NL || frames > l->maxFrames)
        return Fail(HWPA_ERR_INVALID_ARG, "labeler_run: frames outside (24, max_frames]");
    const int nroi = (int)frames + HWPA_VITERBI_LOOKBACK + HWPA_ROI_STITCH;
    const size_t lds = (size_t)((nroi + 15) / 16) * LS * sizeof(uint32_t);
    // Variants: frames per prefetched batch x registers held to 4 waves per SIMD; 0 is the choice
    // by size.
#define HWPA_LABEL_LAUNCH(PB, W)                                                                                   \
    hipLaunchKernelGGL((LabelKernel<PB, W>), dim3(l->lanes), dim3(LS), lds, s, traces, (int)frames, models,        \
                       l->state, l->tb, (int)(l->maxFrames + HWPA_VITERBI_LOOKBACK + NS), labels, latent_out,      \
                       score, l->T, l->roiUpper, l->roiLower)
    const int32_t tuned = TuneGet(kTuneLabel, l->lanes, frames);
    switch (tuned == 0 ? LabelerDefault(l, frames) : tuned) {
    case 1: HWPA_LABEL_LAUNCH(8, 1); break;
    case 2: HWPA_LABEL_LAUNCH(8, 4); break;
    case 3: HWPA_LABEL_LAUNCH(16, 4); break;
    default:
        hipLaunchKernelGGL(LabelQuadKernel, dim3(l->lanes), dim3(4 * LS), lds, s, traces, (int)frames, models,
                           l->state, reinterpret_cast<uint16_t*>(l->tb), (int)(l->maxFrames + HWPA_VITERBI_LOOKBACK),
                           labels, latent_out, score, l->T, l->roiUpper, l->roiLower);
        break;
    }
#undef HWPA_LABEL_LAUNCH
    return CheckLaunch("LabelKernel");
}

}  // namespace hwpa

extern "C" int32_t hwpa_transition_matrix(const hwpa_config* cfg, hwpa_transition* out)
{
    if (!cfg || !out) return hwpa::Fail(HWPA_ERR_INVALID_ARG, "null argument");
    hwpa::BuildTransition(*cfg, *out);
    return HWPA_OK;
}
