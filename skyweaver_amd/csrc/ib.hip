// ib.hip -- incoherent beamformer: weighted Stokes power summed over
// antennas and time-scrunched, for every beamset in one launch.
//
// Reference: IncoherentBeamformer::beamform / icbf_ftpa_general_k,
// cpp/skyweaver/src/IncoherentBeamformer.cu:16-183; oracle
// cpp/skyweaver/test/src/IncoherentBeamformerTester.cu:41-103:
//   P[s][t'][f] = sum_{t in window} sum_a Stokes(v[f][t][0][a], v[f][t][1][a]) * w[s][a]
//   raw = P, out = clamp(rescale(P, offset[s][f], scale[s][f]))
// Unlike the reference kernel (which applies antenna_weights[a] of beamset 0
// to every beamset and caps the antenna count at 64), every beamset uses its
// own weight row and any antenna count works.
//
// The float chain sums in exactly the oracle's order (time ascending, antenna
// ascending, one rounding for the product and one for the sum), so raw powers
// are bit-identical to the oracle for any weights, not only when the sums
// happen to be exact.
//
// Exact fast path (antenna weights all 0 or 1): every term of the float chain
// is an integer, and the terms of Q, U and V are no larger than Stokes I's
// (|2 p0 conj(p1)| <= |p0|^2 + |p1|^2), so while the Stokes I total stays below
// 2^24 every partial sum of any of the four chains is exact and the float
// results equal the integer sums, whatever their order.  The kernel then sums
// with v_dot4_i32_i8 (two antennas of one polarisation per word, masked by the
// beamset's 0/1 weights) and converts once; a workgroup with a Stokes I total
// of 2^24 or more recomputes its outputs with the float chain.
#include "sw_common.hpp"

#include <algorithm>
#include <type_traits>

namespace sw {
namespace {

constexpr int kIbThreads = 256;  // 2^8
constexpr int kSmall = 32;      // antennas x tscrunch of ib_small_kernel's outputs
constexpr int kMaskWords = 64;  // 0/1 weight masks for up to 128 antennas

// 2^24: integers below it are exact in FP32
constexpr int kExact = 1 << 24;

// The power sums of one output: |p0|^2, |p1|^2, and for U and V the halves
// r0 r1 + i0 i1, i0 r1 and r0 i1 of two antennas per word.  The two squares
// saturate (a total past int32 must still read as >= 2^24).
template <int S>
struct IbSums {
    static constexpr bool kU = S == SW_STOKES_U || S == SW_STOKES_IQUV;
    static constexpr bool kV = S == SW_STOKES_V || S == SW_STOKES_IQUV;
    int p0 = 0, p1 = 0, u = 0, v0 = 0, v1 = 0;
    __device__ __forceinline__ void add(uint32_t x0, uint32_t x1, uint32_t m)
    {
        const int a1 = (int)(x1 & m);
        p0 = __builtin_amdgcn_sdot4((int)(x0 & m), (int)x0, p0, true);
        p1 = __builtin_amdgcn_sdot4(a1, (int)x1, p1, true);
        if constexpr(kU) u = __builtin_amdgcn_sdot4((int)x0, a1, u, false);
        if constexpr(kV) {
            // [i, 0] and [0, r] of each antenna (the same for every mask)
            // against x1's [r, i]
            const uint32_t im = __builtin_amdgcn_perm(x0, x0, 0x0C030C01u);
            const uint32_t re = __builtin_amdgcn_perm(x0, x0, 0x020C000Cu);
            v0 = __builtin_amdgcn_sdot4((int)im, a1, v0, false);
            v1 = __builtin_amdgcn_sdot4((int)re, a1, v1, false);
        }
    }
    // Stokes I, at most 2^24 (64 of these sum without overflow)
    __device__ __forceinline__ int total() const { return min(min(p0, kExact) + min(p1, kExact), kExact); }
    // the wanted Stokes parameters but I, exact while I's total is below 2^24
    __device__ __forceinline__ int q() const { return (int)((uint32_t)p0 - (uint32_t)p1); }
    __device__ __forceinline__ int uu() const { return 2 * u; }
    __device__ __forceinline__ int vv() const { return 2 * (int)((uint32_t)v0 - (uint32_t)v1); }
};

// Output o: the powers, and the powers requantised
template <int S>
__device__ __forceinline__ void ib_store(float* raw, int8_t* out, size_t o, const float* power, float off, float sc)
{
    if constexpr(nstokes(S) == 1) {
        raw[o] = power[0];
        out[o] = clamp_i8(rescale<S>(power[0], off, sc));
    } else {
        reinterpret_cast<float4*>(raw)[o] = make_float4(power[0], power[1], power[2], power[3]);
        char4 q;
        q.x = clamp_i8(rescale<SW_STOKES_I>(power[0], off, sc));
        q.y = clamp_i8(rescale<SW_STOKES_Q>(power[1], off, sc));
        q.z = clamp_i8(rescale<SW_STOKES_U>(power[2], off, sc));
        q.w = clamp_i8(rescale<SW_STOKES_V>(power[3], off, sc));
        reinterpret_cast<char4*>(out)[o] = q;
    }
}

// Stokes parameters of antennas a4 ... a4 + 3 of the staged row rb
template <int S>
__device__ __forceinline__ void stokes4(const uint8_t* rb, int nant, int a4, float (&st)[4][nstokes(S)])
{
    // 4 antennas of pol 0 and of pol 1 (8 bytes each, 8-byte aligned)
    const uint2 q0 = *reinterpret_cast<const uint2*>(rb + a4 * 2);
    const uint2 q1 = *reinterpret_cast<const uint2*>(rb + (nant + a4) * 2);
    const uint32_t w0[2] = {q0.x, q0.y};
    const uint32_t w1[2] = {q1.x, q1.y};
#pragma unroll
    for(int j = 0; j < 4; ++j) {
        const uint32_t d0 = w0[j >> 1] >> (16 * (j & 1));
        const uint32_t d1 = w1[j >> 1] >> (16 * (j & 1));
        const float r0 = (float)(int8_t)(d0), i0 = (float)(int8_t)(d0 >> 8);
        const float r1 = (float)(int8_t)(d1), i1 = (float)(int8_t)(d1 >> 8);
        if constexpr(nstokes(S) == 1) {
            st[j][0] = stokes<S>(r0, i0, r1, i1);
        } else {
            st[j][0] = stokes<SW_STOKES_I>(r0, i0, r1, i1);
            st[j][1] = stokes<SW_STOKES_Q>(r0, i0, r1, i1);
            st[j][2] = stokes<SW_STOKES_U>(r0, i0, r1, i1);
            st[j][3] = stokes<SW_STOKES_V>(r0, i0, r1, i1);
        }
    }
}

// lane l's partner in a group of eight: l ^ 7, l ^ 2 or l ^ 1
template <int M>
__device__ __forceinline__ int lane_xor(int v)
{
    static_assert(M == 7 || M == 2 || M == 1, "row_half_mirror, quad_perm");
    return __builtin_amdgcn_mov_dpp(v, M == 7 ? 0x141 : M == 2 ? 0x4E : 0xB1, 0xF, 0xF, true);
}

// One step of LanesSum: with two or more values left a lane gives its
// partner half of them and keeps the half that its bit B selects, else both
// add the one.
template <int M, int B, int N>
__device__ __forceinline__ void lanes_step(int* v, int l)
{
    if constexpr(N == 1) {
        v[0] += lane_xor<M>(v[0]);
    } else {
#pragma unroll
        for(int i = 0; i < N / 2; ++i) {
            const int keep = l & B ? v[N / 2 + i] : v[i], give = l & B ? v[i] : v[N / 2 + i];
            v[i] = keep + lane_xor<M>(give);
        }
    }
}

// The sums of N = 2 or 4 values over groups of N lanes: value l % N in lane l
template <int N>
__device__ __forceinline__ int lanes_deal(int (&v)[N], int l)
{
    static_assert(N == 2 || N == 4, "neighbours of a quad");
    if constexpr(N == 4) lanes_step<2, 2, 4>(v, l);
    lanes_step<1, 1, 2>(v, l);
    return v[0];
}

// The sums of N values (a power of two) over groups of `lanes` (8 ... 64)
// lanes, dealt out: lane l ends with the sums first(l) ... first(l) + N' - 1,
// N' = max(N / 8, 1), in v.  (A tree per value over all lanes, one lane
// storing every value, was a latency of its own each: 64 channels x 65536
// samples x 16 antennas at tscrunch 4, five beamsets, took 226 us, now 141;
// 16 of full Stokes 2.38 ms, now 0.60.)
template <int N>
struct LanesSum {
    static constexpr int kLeft = N < 8 ? 1 : N / 8;
    __device__ static __forceinline__ int first(int l) { return (l & 7) * N / 8; }
    // the lanes that hold sums nobody before them holds
    __device__ static __forceinline__ bool owner(int l) { return l < 8 && (l * N) % 8 < (N < 8 ? N : 8); }
    __device__ static __forceinline__ void run(int* v, int l, int lanes)
    {
        lanes_step<7, 4, N>(v, l);
        lanes_step<2, 2, (N < 2 ? 1 : N / 2)>(v, l);
        lanes_step<1, 1, (N < 4 ? 1 : N / 4)>(v, l);
#pragma unroll
        for(int i = 0; i < kLeft; ++i) {
            if(lanes > 8) v[i] += __builtin_amdgcn_mov_dpp(v[i], 0x128, 0xF, 0xF, true);  // row_ror:8
            if(lanes > 16) v[i] += __builtin_amdgcn_ds_swizzle(v[i], 0x401F);             // lane ^ 16
            if(lanes > 32) v[i] += __shfl_xor(v[i], 32, 64);
        }
    }
};

// A workgroup owns batches = 2^bsh runs of ob = 256 / lanes consecutive outputs
// of one channel, lanes = 2^lsh.  HBM-bound: `lanes` neighbouring lanes share
// an output, each reading 4 W bytes (2 W antennas) of both polarisations of
// every (lanes / chunks)-th row of its scrunch window, up to four rows' loads
// in flight, so that a wave reads whole rows and nothing goes through LDS; the
// lanes' sums meet in LanesSum.  (Staged through LDS by one wave per 64 outputs,
// each lane then summing a whole window, the loads of a row were waited for
// before the sums of it: 64 channels x 16384 samples x 64 antennas, two
// beamsets, took 150 us, IQUV of 16 channels x 32768 samples 206 us.)
template <int S, int SMAX, int W>
__global__ void __launch_bounds__(kIbThreads)
ib_kernel(const uint8_t* __restrict__ ftpa, float* __restrict__ raw, int8_t* __restrict__ out,
          const float* __restrict__ scale, const float* __restrict__ offset,
          const float* __restrict__ antw, int nchans, int nsamps_out, int nant, int tscrunch,
          int nbeamsets, int lsh, int bsh, int csh)
{
    constexpr int NV = nstokes(S);
    using P = typename std::conditional<W == 4, uint4, uint2>::type;
    extern __shared__ uint4 rows[];  // float chain: [ob batches][rowq + 1], then the weights
    const int f    = blockIdx.y;
    const int tid  = threadIdx.x;
    const int lanes = 1 << lsh, batches = 1 << bsh, ob = kIbThreads >> lsh;
    const int tp0  = blockIdx.x * ob * batches;
    const uint8_t* chan = ftpa + (size_t)f * nsamps_out * tscrunch * 4 * nant;

    auto store = [&](int f, int s, int tp, const float* power) {
        ib_store<S>(raw, out, ((size_t)s * nsamps_out + tp) * nchans + f, power, offset[s * nchans + f],
                    scale[s * nchans + f]);
    };

    // ---- exact integer path
    __shared__ uint32_t wmask[SMAX][kMaskWords];  // per word: 0xFFFF per antenna of weight 1
    bool exact = nant <= 2 * kMaskWords;
    if(exact) {
        bool binary = true;
        for(int i = tid; i < nbeamsets * nant / 2; i += kIbThreads) {
            const int sb = i / (nant / 2), j = i % (nant / 2);
            const float w0 = antw[sb * nant + 2 * j], w1 = antw[sb * nant + 2 * j + 1];
            binary = binary && (w0 == 0.0f || w0 == 1.0f) && (w1 == 0.0f || w1 == 1.0f);
            wmask[sb][j] = (w0 != 0.0f ? 0x0000FFFFu : 0u) | (w1 != 0.0f ? 0xFFFF0000u : 0u);
        }
        exact = __syncthreads_and(binary);
    }
    if(exact) {
        const int chunks = nant / (2 * W);        // loads per polarisation of a row
        const int krow   = max(1, lanes / chunks);  // rows an output's lanes read together
        const int l = tid & (lanes - 1);
        bool big = false;
        for(int b = 0; b < batches; ++b) {
            const int tp = tp0 + b * ob + (tid >> lsh);
            IbSums<S> sum[SMAX];
            if(l < krow * chunks && tp < nsamps_out) {
                for(int q = l % chunks; q < chunks; q += lanes) {  // once unless lanes < chunks
                    uint32_t m[SMAX][W];
#pragma unroll
                    for(int s = 0; s < SMAX; ++s)
#pragma unroll
                        for(int j = 0; j < W; ++j) m[s][j] = s < nbeamsets ? wmask[s][q * W + j] : 0u;
                    const P* x = reinterpret_cast<const P*>(chan) + (size_t)tp * tscrunch * 2 * chunks + q;
                    auto row = [&](const P& v0, const P& v1) {
                        const uint32_t* x0 = reinterpret_cast<const uint32_t*>(&v0);
                        const uint32_t* x1 = reinterpret_cast<const uint32_t*>(&v1);
#pragma unroll
                        for(int s = 0; s < SMAX; ++s)
                            if(s < nbeamsets)
#pragma unroll
                                for(int j = 0; j < W; ++j) sum[s].add(x0[j], x1[j], m[s][j]);
                    };
                    int tt = l / chunks;
                    for(; tt + 3 * krow < tscrunch; tt += 4 * krow) {
                        P v[8];
#pragma unroll
                        for(int k = 0; k < 4; ++k) {
                            const P* r = x + (size_t)(tt + k * krow) * 2 * chunks;
                            v[2 * k]     = r[0];
                            v[2 * k + 1] = r[chunks];
                        }
#pragma unroll
                        for(int k = 0; k < 4; ++k) row(v[2 * k], v[2 * k + 1]);
                    }
                    for(; tt < tscrunch; tt += krow) {
                        const P* r = x + (size_t)tt * 2 * chunks;
                        row(r[0], r[chunks]);
                    }
                }
            }
            // the lanes' sums meet, and a lane finishes its share of the beamsets
            using L = LanesSum<SMAX>;
            int v[NV + (S == SW_STOKES_I || NV == 4 ? 0 : 1)][SMAX];  // I, then the others wanted
#pragma unroll
            for(int s = 0; s < SMAX; ++s) {
                v[0][s] = sum[s].total();
                if constexpr(S == SW_STOKES_Q || NV == 4) v[1][s] = sum[s].q();
                if constexpr(S == SW_STOKES_U) v[1][s] = sum[s].uu();
                if constexpr(S == SW_STOKES_V) v[1][s] = sum[s].vv();
                if constexpr(NV == 4) {
                    v[2][s] = sum[s].uu();
                    v[3][s] = sum[s].vv();
                }
            }
            constexpr int NVI = sizeof(v) / sizeof(v[0]);
#pragma unroll
            for(int k = 0; k < NVI; ++k) L::run(v[k], l, lanes);
#pragma unroll
            for(int i = 0; i < L::kLeft; ++i) {
                big = big || v[0][i] >= kExact;
                if(L::owner(l) && L::first(l) + i < nbeamsets && tp < nsamps_out) {
                    float power[NV];
#pragma unroll
                    for(int k = 0; k < NV; ++k) power[k] = (float)v[NVI - NV + k][i];
                    store(f, L::first(l) + i, tp, power);
                }
            }
        }
        if(!__syncthreads_or(big)) return;
    }

    // ---- float chain: the rows t' ts + tt (one per output) staged in LDS with
    // coalesced 16-byte loads, beside the weights.  Bound by its serial adds
    // (each waits for the one before), so it wants many outputs in flight and
    // no thread idle: the beamsets are dealt to the threads beside the
    // outputs, thread tid summing output tid mod run of the beamsets
    // tid / run + G k, antennas ascending.  Weights other than 0 and 1 are the
    // same for every workgroup: then the first of them take 2^csh outputs
    // each, counted over all channels, and the others have none.
    // (One thread per output summing every beamset, 4 to 64 outputs a
    // workgroup, left most of it idle and spilled scalar registers on the
    // weights: 64 channels x 16384 samples x 64 antennas at tscrunch 16, five
    // beamsets of weights other than 0 and 1, took 1.10 ms, now 0.15; with 144
    // antennas 9.4 ms, now 0.49; 65536 samples x 16 antennas at tscrunch 4,
    // full Stokes, five beamsets, with at most 64 outputs a workgroup 327 us,
    // now 204.)
    const int rsh = exact ? 8 - lsh + bsh : csh, run = 1 << rsh;
    int fc = f, t0 = tp0;
    if(!exact) {
        const unsigned per = ((unsigned)nsamps_out + run - 1) >> csh;
        const unsigned w = blockIdx.y * gridDim.x + blockIdx.x;
        if(w >= per * nchans) return;  // whole workgroup, before any barrier
        fc = w / per;
        t0 = (int)(w % per) << csh;
    }
    const int nrows = min(run, nsamps_out - t0);
    const int G = kIbThreads >> rsh;  // threads per output
    const int o = tid & (run - 1), s0 = tid >> rsh;
    const bool active = o < nrows && s0 < nbeamsets;
    // beamsets of the wave's first thread: no thread of it has more
    const int kn = __builtin_amdgcn_readfirstlane((nbeamsets - s0 + G - 1) >> (8 - rsh));
    const int rowq = nant / 4;  // 16-byte pieces per row: 4 nant bytes
    const int ldsq = rowq + 1;
    const uint4* chan16 = reinterpret_cast<const uint4*>(ftpa + (size_t)fc * nsamps_out * tscrunch * 4 * nant);
    float* wl = reinterpret_cast<float*>(rows + run * ldsq);  // [beamset][antenna]
    for(int i = tid; i < nbeamsets * nant; i += kIbThreads) wl[i] = antw[i];
    float power[SMAX][NV];
#pragma unroll
    for(int k = 0; k < SMAX; ++k)
#pragma unroll
        for(int v = 0; v < NV; ++v) power[k][v] = 0.0f;
    for(int tt = 0; tt < tscrunch; ++tt) {
        __syncthreads();
        for(int i = tid; i < nrows * rowq; i += kIbThreads) {
            const int r = i / rowq, q = i % rowq;
            rows[r * ldsq + q] = chan16[((size_t)(t0 + r) * tscrunch + tt) * rowq + q];
        }
        __syncthreads();
        if(active) {
            const uint8_t* rb = reinterpret_cast<const uint8_t*>(rows + o * ldsq);
            for(int a4 = 0; a4 < nant; a4 += 4) {
                float st[4][NV];
                stokes4<S>(rb, nant, a4, st);
#pragma unroll
                for(int k = 0; k < SMAX; ++k)
                    if(k == 0 || k < kn) {  // uniform; a thread past the beamsets takes any weights
                        const float4 w =
                            *reinterpret_cast<const float4*>(wl + min(s0 + G * k, nbeamsets - 1) * nant + a4);
#pragma unroll
                        for(int j = 0; j < 4; ++j)
#pragma unroll
                            for(int v = 0; v < NV; ++v)
                                power[k][v] += st[j][v] * (j == 0 ? w.x : j == 1 ? w.y : j == 2 ? w.z : w.w);
                    }
            }
        }
    }
    if(!active) return;
#pragma unroll
    for(int k = 0; k < SMAX; ++k)
        if(s0 + G * k < nbeamsets) store(fc, s0 + G * k, t0 + o, power[k]);
}

// Outputs of few rows and antennas (see launch_ib): one wave per 64 outputs of
// one channel, a lane per output, the rows staged as for the float chain.  Sums
// are few and dealing them to neighbouring lanes costs more than it saves: 64
// channels x 65536 samples x 16 antennas at tscrunch 1 take 91 us so and 183
// in ib_kernel.  Stokes I with weights of 0 and 1 in integers (the
// totals are at most 2^21), the rest as the float chain.
template <int S, int SMAX>
__global__ void __launch_bounds__(64)
ib_small_kernel(const uint8_t* __restrict__ ftpa, float* __restrict__ raw, int8_t* __restrict__ out,
                const float* __restrict__ scale, const float* __restrict__ offset,
                const float* __restrict__ antw, int nchans, int nsamples, int nant, int tscrunch,
                int nbeamsets)
{
    constexpr int NV = nstokes(S);
    extern __shared__ uint4 rows[];  // [64][rowq + 1]
    __shared__ uint32_t wmask[SMAX][kSmall / 2];  // per word: 0xFFFF per antenna of weight 1
    const int f    = blockIdx.y;
    const int lane = threadIdx.x;
    const int nsamps_out = nsamples / tscrunch;
    const int tp0  = blockIdx.x * 64;
    const int rowq = nant / 4;  // 16-byte pieces per row: 4 nant bytes
    const int ldsq = rowq + 1;
    const int nrows = min(64, nsamps_out - tp0);
    const uint4* chan = reinterpret_cast<const uint4*>(ftpa + (size_t)f * nsamples * 4 * nant);
    bool exact = false;
    if constexpr(S == SW_STOKES_I) {
        bool binary = true;
        for(int i = lane; i < nbeamsets * nant / 2; i += 64) {
            const int sb = i / (nant / 2), j = i % (nant / 2);
            const float w0 = antw[sb * nant + 2 * j], w1 = antw[sb * nant + 2 * j + 1];
            binary = binary && (w0 == 0.0f || w0 == 1.0f) && (w1 == 0.0f || w1 == 1.0f);
            wmask[sb][j] = (w0 != 0.0f ? 0x0000FFFFu : 0u) | (w1 != 0.0f ? 0xFFFF0000u : 0u);
        }
        exact = __syncthreads_and(binary);
    }
    float power[SMAX][NV];
    int isum[SMAX];
#pragma unroll
    for(int s = 0; s < SMAX; ++s) {
        isum[s] = 0;
#pragma unroll
        for(int k = 0; k < NV; ++k) power[s][k] = 0.0f;
    }
    for(int tt = 0; tt < tscrunch; ++tt) {
        __syncthreads();
        for(int i = lane; i < nrows * rowq; i += 64) {
            const int r = i / rowq, q = i % rowq;
            rows[r * ldsq + q] = chan[((size_t)(tp0 + r) * tscrunch + tt) * rowq + q];
        }
        __syncthreads();
        if(lane >= nrows) continue;
        if(exact) {
            const int hw = nant / 2;  // words per polarisation
            const uint32_t* rw = reinterpret_cast<const uint32_t*>(rows + lane * ldsq);
#pragma unroll
            for(int s = 0; s < SMAX; ++s)
                if(s < nbeamsets)
                    for(int j = 0; j < hw; ++j) {
                        const int m = (int)wmask[s][j];
                        const int x0 = (int)rw[j], x1 = (int)rw[hw + j];
                        isum[s] = __builtin_amdgcn_sdot4(x0 & m, x0, isum[s], false);
                        isum[s] = __builtin_amdgcn_sdot4(x1 & m, x1, isum[s], false);
                    }
        } else {
            for(int a4 = 0; a4 < nant; a4 += 4) {
                float st[4][NV];
                stokes4<S>(reinterpret_cast<const uint8_t*>(rows + lane * ldsq), nant, a4, st);
#pragma unroll
                for(int j = 0; j < 4; ++j)
#pragma unroll
                    for(int s = 0; s < SMAX; ++s)
                        if(s < nbeamsets) {
                            const float w = antw[s * nant + a4 + j];
#pragma unroll
                            for(int k = 0; k < NV; ++k) power[s][k] += st[j][k] * w;
                        }
            }
        }
    }
    if(lane >= nrows) return;
#pragma unroll
    for(int s = 0; s < SMAX; ++s)
        if(s < nbeamsets) {
            if(exact) power[s][0] = (float)isum[s];
            ib_store<S>(raw, out, ((size_t)s * nsamps_out + tp0 + lane) * nchans + f, power[s],
                        offset[s * nchans + f], scale[s * nchans + f]);
        }
}

// Time-major input (the coherent dedisperser's ring): sample t of column
// c = p A + a of channel f at ring + ((f 2A + c) ld + w0 + t) 2.  0/1 antenna
// weights only.  A workgroup owns 256 / WA outputs t' of channel f; with WA = 4
// its four waves take every fourth antenna, a lane reading its output's ts
// consecutive samples of both polarisations (64 lanes read 64 ts 2 contiguous
// bytes) and adding the antenna's integer sums to the beamsets that weight it
// 1; the waves' sums meet in LDS.  HBM-bound (a workgroup per 256 outputs, one
// lane summing all antennas, left half of the CUs idle at 16 channels x 2048
// outputs; ib_beamform_tm has the rule).  As in ib_kernel the integer totals
// equal the oracle's float chains while Stokes I is below 2^24; a lane at or
// above it recomputes its outputs with the float chains in the oracle's order
// (time, then antenna ascending).
//
// L: 16-byte loads of L neighbouring lanes make up an output's window (ts = 8 L;
// with L = 1 a lane takes all of a window of 8 n samples); 0: 2-byte loads.
// With L > 1 a load of the wave covers whole lines, the windows of 64 / L
// outputs; the L lanes' sums of L such loads are dealt out, so that each lane
// ends with one output's, and the next antenna's loads are in flight meanwhile.
// (A lane that took a window of 32 samples by itself left 64 lines half used by
// each load, and where the columns' pitch is a large power of two these did not
// stay in the cache: full Stokes of 16 antennas x 16 channels x 131072 samples
// took 107 us, now 30; 64 x 8 x 16384 22.4, now 13.8; at tscrunch 16 43 and 30,
// 16.0 and 12.7.  Without the loads ahead the last is 14.4, and with each load
// summed where it was issued 30.8 at tscrunch 32.)
constexpr int kTmMaxAnts = 128;

template <int S, int SMAX, int L, int WA>
__global__ void __launch_bounds__(kIbThreads)
ib_tm_kernel(const uint8_t* __restrict__ ring, long ld, long w0, float* __restrict__ raw,
             int8_t* __restrict__ out, const float* __restrict__ scale, const float* __restrict__ offset,
             const float* __restrict__ antw, int nchans, int nsamples, int nant, int ts, int nbeamsets)
{
    constexpr int NV = nstokes(S), OUT = kIbThreads / WA;
    __shared__ uint8_t antb[SMAX][kTmMaxAnts];  // weight (0/1) of antenna a in beamset s
    __shared__ int red[WA > 1 ? WA : 1][4][OUT];
    for(int i = threadIdx.x; i < nbeamsets * nant; i += kIbThreads)
        antb[i / nant][i % nant] = antw[i] != 0.0f ? 1 : 0;
    __syncthreads();
    const int f = blockIdx.y;
    const int lane = threadIdx.x % OUT, wave = threadIdx.x / OUT;
    const int nsamps_out = nsamples / ts;
    // the lane's output, and with L > 1 the outputs first + j 64 / L whose
    // piece l % L it loads
    constexpr int LL = L > 1 ? L : 1, G = 64 / LL;
    const int l = threadIdx.x % 64, first = blockIdx.x * OUT + lane - l + l / LL;
    const int tp = first + l % LL * G;
    const bool active = tp < nsamps_out;
    const uint8_t* chan = ring + ((size_t)f * 2 * nant * ld + w0) * 2 + l % LL * 16;
    const uint8_t* base = ring + ((size_t)f * 2 * nant * ld + w0 + (size_t)(active ? tp : 0) * ts) * 2;
    int si[SMAX], sq[SMAX], su[SMAX], sv[SMAX];
#pragma unroll
    for(int s = 0; s < SMAX; ++s) si[s] = sq[s] = su[s] = sv[s] = 0;
    uint4 ny[LL], nz[LL];
    auto fetch = [&](int a) {
#pragma unroll
        for(int j = 0; j < L; ++j) {
            const int o = first + j * G < nsamps_out ? first + j * G : 0;
            const uint8_t* x = chan + ((size_t)a * ld + (size_t)o * (8 * L)) * 2;
            ny[j] = *reinterpret_cast<const uint4*>(x);
            nz[j] = *reinterpret_cast<const uint4*>(x + (size_t)nant * ld * 2);
        }
    };
    if constexpr(L > 1)
        if(wave < nant) fetch(wave);
    constexpr int U = L > 1 ? 1 : WA > 1 ? 2 : 4;
#pragma unroll U
    for(int a = wave; a < nant; a += WA) {
        const uint8_t* x0 = base + (size_t)a * ld * 2;
        const uint8_t* x1 = base + (size_t)(nant + a) * ld * 2;
        IbSums<S> c;
        int i = 0, q = 0, u = 0, v = 0;  // the antenna's sums of the lane's output
        if constexpr(L > 1) {
            uint4 y[L], z[L];
#pragma unroll
            for(int j = 0; j < L; ++j) y[j] = ny[j], z[j] = nz[j];
            fetch(a + WA < nant ? a + WA : a);
            __builtin_amdgcn_sched_barrier(0);
            int vi[L], vq[L], vu[L], vv[L];
#pragma unroll
            for(int j = 0; j < L; ++j) {
                IbSums<S> b;
                b.add(y[j].x, z[j].x, ~0u);
                b.add(y[j].y, z[j].y, ~0u);
                b.add(y[j].z, z[j].z, ~0u);
                b.add(y[j].w, z[j].w, ~0u);
                vi[j] = b.p0 + b.p1;  // at most 2^19
                vq[j] = b.q(), vu[j] = b.uu(), vv[j] = b.vv();
            }
            i = lanes_deal<L>(vi, l);
            if constexpr(S == SW_STOKES_Q || NV == 4) q = lanes_deal<L>(vq, l);
            if constexpr(S == SW_STOKES_U || NV == 4) u = lanes_deal<L>(vu, l);
            if constexpr(S == SW_STOKES_V || NV == 4) v = lanes_deal<L>(vv, l);
        } else if constexpr(L == 1) {  // ts % 8 == 0: 16-byte aligned runs
            for(int k = 0; k < ts * 2; k += 16) {
                const uint4 v = *reinterpret_cast<const uint4*>(x0 + k), w = *reinterpret_cast<const uint4*>(x1 + k);
                c.add(v.x, w.x, ~0u);
                c.add(v.y, w.y, ~0u);
                c.add(v.z, w.z, ~0u);
                c.add(v.w, w.w, ~0u);
            }
        } else {
            for(int k = 0; k < ts; ++k)
                c.add(*reinterpret_cast<const uint16_t*>(x0 + 2 * k), *reinterpret_cast<const uint16_t*>(x1 + 2 * k), ~0u);
        }
        if constexpr(L <= 1) {
            i = WA > 1 ? c.total() : c.p0 + c.p1;
            q = c.q(), u = c.uu(), v = c.vv();
        }
#pragma unroll
        for(int s = 0; s < SMAX; ++s)
            if(s < nbeamsets && antb[s][a]) {
                si[s] += i;  // at most 32 of 2^24, or 2^30 in all (the rule)
                if constexpr(S == SW_STOKES_Q || NV == 4) sq[s] += q;
                if constexpr(S == SW_STOKES_U || NV == 4) su[s] += u;
                if constexpr(S == SW_STOKES_V || NV == 4) sv[s] += v;
            }
    }
#pragma unroll
    for(int s = 0; s < SMAX; ++s) {
        if(s < nbeamsets) {  // uniform
            int t[4] = {si[s], sq[s], su[s], sv[s]};
            if constexpr(WA > 1) {
                if(s) __syncthreads();
                red[wave][0][lane] = min(si[s], kExact);
                if constexpr(S != SW_STOKES_I) {
                    red[wave][1][lane] = sq[s];
                    red[wave][2][lane] = su[s];
                    red[wave][3][lane] = sv[s];
                }
                __syncthreads();
            }
            if(wave == 0 && active) {
                if constexpr(WA > 1) {
#pragma unroll
                    for(int k = 0; k < (S == SW_STOKES_I ? 1 : 4); ++k) {
                        t[k] = 0;
#pragma unroll
                        for(int w = 0; w < WA; ++w) t[k] += red[w][k][lane];
                    }
                }
                float power[NV];
                if constexpr(NV == 4) {
#pragma unroll
                    for(int k = 0; k < 4; ++k) power[k] = (float)t[k];
                } else {
                    power[0] = (float)t[S == SW_STOKES_I ? 0 : S == SW_STOKES_Q ? 1 : S == SW_STOKES_U ? 2 : 3];
                }
                if(t[0] >= kExact) {  // the oracle's float chains
#pragma unroll
                    for(int k = 0; k < NV; ++k) power[k] = 0.0f;
                    for(int tt = 0; tt < ts; ++tt)
                        for(int a = 0; a < nant; ++a) {
                            const uint16_t d0 = *reinterpret_cast<const uint16_t*>(base + ((size_t)a * ld + tt) * 2);
                            const uint16_t d1 = *reinterpret_cast<const uint16_t*>(base + ((size_t)(nant + a) * ld + tt) * 2);
                            const float r0 = (float)(int8_t)d0, i0 = (float)(int8_t)(d0 >> 8);
                            const float r1 = (float)(int8_t)d1, i1 = (float)(int8_t)(d1 >> 8);
                            const float w = antw[s * nant + a];
                            if constexpr(NV == 1) {
                                power[0] += stokes<S>(r0, i0, r1, i1) * w;
                            } else {
                                power[0] += stokes<SW_STOKES_I>(r0, i0, r1, i1) * w;
                                power[1] += stokes<SW_STOKES_Q>(r0, i0, r1, i1) * w;
                                power[2] += stokes<SW_STOKES_U>(r0, i0, r1, i1) * w;
                                power[3] += stokes<SW_STOKES_V>(r0, i0, r1, i1) * w;
                            }
                        }
                }
                ib_store<S>(raw, out, ((size_t)s * nsamps_out + tp) * nchans + f, power, offset[s * nchans + f],
                            scale[s * nchans + f]);
            }
        }
    }
}

template <int S>
int launch_ib(const uint8_t* ftpa, float* raw, int8_t* out, const float* scale,
              const float* offset, const float* antw, const sw_bf_dims& d, hipStream_t st)
{
    const int nout = d.nsamples / d.tscrunch;
    // where ib_small_kernel is the faster, one beamset over all 64 channels:
    // 16384 samples x 4 antennas at tscrunch 1 14.1 us and 37.8, 16 antennas
    // 18.7 and 41.8; 8192 samples x 16 antennas at tscrunch 2 8.5 and 13.6, x
    // 32 at 1 17.1 and 23.3.  Not with more rows a window (65536 samples x 8
    // antennas at tscrunch 4: 77 and 43) or few outputs, for which ib_kernel
    // finds more lanes (8 channels x 4096 samples x 16 antennas at tscrunch 2,
    // sixteen beamsets: 11.5 and 7.6)
    const int window = d.nantennas * d.tscrunch;
    const long waves = (long)((nout + 63) / 64) * d.nchans;
    if((window <= kSmall / 2 && waves >= 512) || (window <= kSmall && d.tscrunch <= 2 && waves >= 2048)) {
        const dim3 grid((unsigned)((nout + 63) / 64), d.nchans);
        const size_t lds = (size_t)64 * (d.nantennas / 4 + 1) * 16;
#define SW_IB_LAUNCH(SM)                                                                                           \
    hipLaunchKernelGGL((ib_small_kernel<S, SM>), grid, dim3(64), lds, st, ftpa, raw, out, scale, offset, antw,     \
                       d.nchans, d.nsamples, d.nantennas, d.tscrunch, d.nbeamsets);
        if(d.nbeamsets <= 1) {
            SW_IB_LAUNCH(1)
        } else if(d.nbeamsets <= 4) {
            SW_IB_LAUNCH(4)
        } else if(d.nbeamsets <= 8) {
            SW_IB_LAUNCH(8)
        } else {
            SW_IB_LAUNCH(16)
        }
#undef SW_IB_LAUNCH
        SW_LAUNCH_CHECK();
        return SW_OK;
    }
    const bool w4 = d.nantennas % 8 == 0;  // 16-byte loads, else 8-byte
    const int chunks = d.nantennas / (w4 ? 8 : 4);
    // 8 lanes per output (a row of 64 antennas' polarisation at 16 bytes a
    // lane), more where a row takes more loads; then, while the chip is not
    // filled four times over with workgroups, more lanes with fewer rows
    // each, down to the four rows a lane has in flight
    int lanes = 8;
    while(lanes < 64 && lanes < chunks) lanes *= 2;
    auto groups = [&](int ob) { return (long)((nout + ob - 1) / ob) * d.nchans; };
    while(lanes < 64 && groups(kIbThreads / lanes) < 1024 && (long)d.tscrunch * chunks >= 8L * lanes) lanes *= 2;
    // 64 outputs per workgroup where enough workgroups are left
    int batches = groups(64) >= 2048 ? 64 * lanes / kIbThreads : 1;
    if(nout > 1 << 29) batches = lanes;  // 256: the grid's threads stay below 2^32
    // LDS of the float chain for n outputs at a time: rows and weights
    auto chain_lds = [&](int n) {
        return (size_t)n * (d.nantennas / 4 + 1) * 16 + (size_t)d.nbeamsets * d.nantennas * 4;
    };
    // the float chain's outputs per workgroup where it runs alone: a thread
    // per output, fewer outputs (and a thread for some of the beamsets) while
    // few workgroups fit a CU's LDS or the chip is not filled four times over
    int nchain = 256;
    while(nchain > 4 && (groups(nchain) < 1024 || chain_lds(nchain) > (size_t)(nchain > 64 ? 25 : 72) << 10)) nchain /= 2;
    if(d.nantennas > 2 * kMaskWords) {  // it does
        lanes   = kIbThreads / nchain;
        batches = 1;
    }
    const int ob = kIbThreads / lanes;
    nchain = std::max(nchain, ob * batches);  // the workgroups suffice
    const dim3 grid((unsigned)((nout + ob * batches - 1) / (ob * batches)), d.nchans);
    const size_t lds = chain_lds(nchain);
    auto log2i = [](int v) { return __builtin_ctz((unsigned)v); };  // of a power of two
#define SW_IB_LAUNCH_W(SM, W)                                                                                      \
    hipLaunchKernelGGL((ib_kernel<S, SM, W>), grid, dim3(kIbThreads), lds, st, ftpa, raw, out, scale, offset, antw, \
                       d.nchans, nout, d.nantennas, d.tscrunch, d.nbeamsets, log2i(lanes), log2i(batches),         \
                       log2i(nchain))
#define SW_IB_LAUNCH(SM)       \
    if(w4)                     \
        SW_IB_LAUNCH_W(SM, 4); \
    else                       \
        SW_IB_LAUNCH_W(SM, 2);
    if(d.nbeamsets <= 1) {
        SW_IB_LAUNCH(1)
    } else if(d.nbeamsets <= 2) {
        SW_IB_LAUNCH(2)
    } else if(d.nbeamsets <= 4) {
        SW_IB_LAUNCH(4)
    } else if(d.nbeamsets <= 8) {
        SW_IB_LAUNCH(8)
    } else {
        SW_IB_LAUNCH(16)
    }
#undef SW_IB_LAUNCH
#undef SW_IB_LAUNCH_W
    SW_LAUNCH_CHECK();
    return SW_OK;
}

} // namespace

// Incoherent beam from the dedisperser's time-major ring (see ib_tm_kernel):
// Stokes I or IQUV, 0/1 antenna weights, d.nantennas <= 128.
int ib_beamform_tm(const void* d_ring, long ld, long w0, float* d_raw, void* d_out, const float* d_scale,
                   const float* d_offset, const float* d_ant_weights, const sw_bf_dims& d, hipStream_t st)
{
    SW_CHECK_ARG(d_ring && d_raw && d_out && d_scale && d_offset && d_ant_weights, "null buffer");
    SW_CHECK_ARG((d.stokes == SW_STOKES_I || d.stokes == SW_STOKES_IQUV) && d.nantennas <= kTmMaxAnts,
                 "time-major IB: Stokes I or IQUV, <= 128 antennas");
    SW_CHECK_ARG(d.nbeamsets > 0 && d.nbeamsets <= 16 && d.nchans > 0 && d.nchans <= 65535, "bad dimensions");
    SW_CHECK_ARG(d.tscrunch > 0 && d.nsamples % d.tscrunch == 0, "nsamples must be a multiple of tscrunch");
    SW_CHECK_ARG((reinterpret_cast<uintptr_t>(d_ring) & 15) == 0 && ld % 8 == 0 && w0 % 8 == 0,
                 "ring must be 16-byte aligned with 8-sample aligned rows");
    const int nout = d.nsamples / d.tscrunch;
    const bool v16 = d.tscrunch % 8 == 0;
    // 256 outputs per workgroup, no shared antennas, where the rows come from
    // HBM (more than the 256 MB behind L2 hold) and a workgroup's run of a
    // column is long: the four waves then read one run of 512 tscrunch bytes
    // instead of four of 128.  48 antennas x 32 channels x 65536 samples at
    // tscrunch 8 99 us shared, 85 so, at 16 97 and 82, at 32 96 and 83; 32 x 32 x
    // 65536, full Stokes, 67 and 53 at 16, 71 and 50 at 32.  Shared where that
    // leaves fewer workgroups than CUs or the samples stay on the chip (48 x 16
    // x 65536 at 8 40 and 47), at other tscrunches (48 x 64 x 40960 at 4: 182
    // and 241), and for more than four beamsets where lanes share an output and
    // the columns lie at no large power of two (16 x 64 x 73728, full Stokes,
    // eight: 113 and 142 at 16, 102 and 121 at 32; 48 x 64 x 40960 136 and 150,
    // 132 and 146)
    const long groups = (long)((nout + kIbThreads - 1) / kIbThreads) * d.nchans;
    const long bytes = 4L * d.nantennas * d.nchans * d.nsamples;
    const int dealt = d.tscrunch == 16 ? 2 : d.tscrunch == 32 ? 4 : 1;  // lanes per output
    const bool share = !(v16 && groups >= 256 && groups <= 2048 && bytes >= 256L << 20 &&
                         (d.nsamples >= 32768 || bytes > 384L << 20) &&
                         (dealt == 1 || d.nbeamsets <= 4 || d.nsamples % 16384 == 0) &&
                         d.tscrunch <= 16384 / d.nantennas);  // totals of at most 2^30
    auto* in = static_cast<const uint8_t*>(d_ring);
    auto* out = static_cast<int8_t*>(d_out);
    const int ob = share ? kIbThreads / 4 : kIbThreads;
    const dim3 grid((unsigned)((nout + ob - 1) / ob), d.nchans);
#define SW_IBT_L(S, SM, V, WA)                                                                                       \
    hipLaunchKernelGGL((ib_tm_kernel<S, SM, V, WA>), grid, dim3(kIbThreads), 0, st, in, ld, w0, d_raw, out, d_scale, \
                       d_offset, d_ant_weights, d.nchans, d.nsamples, d.nantennas, d.tscrunch, d.nbeamsets)
#define SW_IBT_V(S, SM)              \
    if(!v16)                         \
        SW_IBT_L(S, SM, 0, 4);       \
    else if(dealt == 2 && !share)    \
        SW_IBT_L(S, SM, 2, 1);       \
    else if(dealt == 4 && !share)    \
        SW_IBT_L(S, SM, 4, 1);       \
    else if(!share)                  \
        SW_IBT_L(S, SM, 1, 1);       \
    else if(dealt == 2)              \
        SW_IBT_L(S, SM, 2, 4);       \
    else if(dealt == 4)              \
        SW_IBT_L(S, SM, 4, 4);       \
    else                             \
        SW_IBT_L(S, SM, 1, 4);
#define SW_IBT(SM)                   \
    if(d.stokes == SW_STOKES_I) {    \
        SW_IBT_V(SW_STOKES_I, SM)    \
    } else {                         \
        SW_IBT_V(SW_STOKES_IQUV, SM) \
    }
    if(d.nbeamsets <= 1) {
        SW_IBT(1)
    } else if(d.nbeamsets <= 4) {
        SW_IBT(4)
    } else if(d.nbeamsets <= 8) {
        SW_IBT(8)
    } else {
        SW_IBT(16)
    }
#undef SW_IBT
#undef SW_IBT_V
#undef SW_IBT_L
    SW_LAUNCH_CHECK();
    return SW_OK;
}

} // namespace sw

extern "C" int sw_ib_beamform(const void* d_ftpa, float* d_raw, void* d_out,
                              const float* d_scale, const float* d_offset,
                              const float* d_ant_weights, const sw_bf_dims* dims,
                              void* stream)
{
    SW_CHECK_ARG(dims, "null dims");
    const sw_bf_dims& d = *dims;
    SW_CHECK_ARG(d_ftpa && d_raw && d_out && d_scale && d_offset && d_ant_weights, "null buffer");
    SW_CHECK_ARG(d.nbeamsets > 0, "Number of beamsets must be greater than zero");
    SW_CHECK_ARG(d.nbeamsets <= 16, "at most 16 beamsets are supported");
    SW_CHECK_ARG(d.nchans > 0 && d.nchans <= 65535, "bad channel count");
    SW_CHECK_ARG(d.nantennas > 0 && d.nantennas % 4 == 0, "antenna count must be a multiple of 4");
    SW_CHECK_ARG(d.tscrunch > 0 && d.nsamples > 0 && d.nsamples % d.tscrunch == 0,
                 "nsamples must be a positive multiple of tscrunch");
    SW_CHECK_ARG(d.stokes >= SW_STOKES_I && d.stokes <= SW_STOKES_IQUV, "bad stokes mode");
    SW_CHECK_ARG((reinterpret_cast<uintptr_t>(d_ftpa) & 15) == 0, "input must be 16-byte aligned");
    SW_CHECK_ARG(d.nantennas <= 512, "at most 512 antennas");
    auto* in  = static_cast<const uint8_t*>(d_ftpa);
    auto* out = static_cast<int8_t*>(d_out);
    hipStream_t st = sw::as_stream(stream);
    switch(d.stokes) {
    case SW_STOKES_I: return sw::launch_ib<SW_STOKES_I>(in, d_raw, out, d_scale, d_offset, d_ant_weights, d, st);
    case SW_STOKES_Q: return sw::launch_ib<SW_STOKES_Q>(in, d_raw, out, d_scale, d_offset, d_ant_weights, d, st);
    case SW_STOKES_U: return sw::launch_ib<SW_STOKES_U>(in, d_raw, out, d_scale, d_offset, d_ant_weights, d, st);
    case SW_STOKES_V: return sw::launch_ib<SW_STOKES_V>(in, d_raw, out, d_scale, d_offset, d_ant_weights, d, st);
    default: return sw::launch_ib<SW_STOKES_IQUV>(in, d_raw, out, d_scale, d_offset, d_ant_weights, d, st);
    }
}
