// idisp.hip -- incoherent (post-detection) dedispersion of TFB powers on the
// GPU, and the DedispersionPlan block parser.
//
// Reference: IncoherentDedisperser::prepare / dedisperse,
// cpp/skyweaver/src/IncoherentDedisperser.cu:36-125, with DMSampleDelay
// (cpp/skyweaver/dedispersion_utils.cuh:19-40):
//   delta[d][f] = (int)(K dm_d (1/f_0^2 - 1/f^2) / tsamp + 0.5), f_0 = lowest channel,
//   tsamp = cb_tscrunch / (bandwidth / nchans)
//   out[t'][d][b] = (int8)clamp(sum_{s<ts} sum_f in[D + t' ts + s - delta[d][f]][f][b]
//                               / (float)sqrt(F ts))
// with D = max delta and t' < (T - D) / ts.  The sums are exact integers, so
// the summation order is free; the division and the truncating clamp are the
// reference's.
//
// Kernel design: a workgroup owns 64 words (256 bytes) of a (t, f) row,
// TT output samples and a tile of up to 4 DPW consecutive DMs (one wave per
// DM residue).  For every channel it stages the union of the rows its DMs
// read into LDS, biased by XOR 0x80 so every byte is an unsigned x + 128; each
// lane then adds its word into two registers of 16-bit lanes (even and odd
// bytes), i.e. four beam sums per two integer adds.  The 16-bit lanes hold
// at most 256 biased bytes; longer sums (nchans * ts > 256) are flushed into
// 32-bit accumulators.
//
// Matrix-core form (idisp_tile, used whenever nchans % 4 == 0 and the rows of
// one DM fit the stage): one DM's channel sum is a chain of
// v_mfma_i32_16x16x64_i8 products.  The B operand carries data: lane
// (n, g) = (l % 16, l / 16) holds the 16 beam bytes [b0, b0 + 16) of channel
// f0 + g at the input row of output sample n.  The A operand is a constant
// selector, row m holding a single 1 at byte m of every k-group, so
// C[m][n] = sum over g of beam b0 + m of channel f0 + g at sample n: four
// channels x 16 beams x 16 samples per instruction, summed exactly in int32.
// It runs as idisp_dma_kernel (tscrunch <= 2, 32 output samples per
// workgroup) and idisp_mfma_kernel (tscrunch 3-8, 16 samples).
#include "sw_common.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <sstream>
#include <string>
#include <type_traits>
#include <vector>

struct sw_idisp {
    int nchans = 0, ndms = 0, tscrunch = 1;
    int max_delay = 0;
    float scale = 1.0f;
    std::vector<float> dms;
    std::vector<int> delays;          // [D][F]
    // device tiling
    int dpw = 2, tt = 16, rows_cap = 0;
    bool wide = false;
    bool mfma = false;                // matrix-core kernel (else the 16-bit-lane one)
    bool small = false;               // its small form: 8 waves, two workgroups per CU
    std::vector<int2> tiles;          // (first DM, count)
    int* d_delays = nullptr;
    uint8_t* d_rel = nullptr;         // matrix-core form: [ntiles][F][waves] delta_max - delta
    int2* d_span = nullptr;           // [ntiles][F] (delta_min, delta_max)
    int2* d_tiles = nullptr;
};

namespace sw {
namespace {

constexpr double kDmConstHzS = 4.148806423e15;  // Hz^2 pc^-1 cm^3 s

// one step of 16-bit-lane accumulation of a biased word
__device__ __forceinline__ void id_add(uint32_t w, uint32_t& e, uint32_t& o)
{
    e += w & 0x00FF00FFu;
    o += (w >> 8) & 0x00FF00FFu;
}

__device__ __forceinline__ int8_t id_quant(int32_t sum, float scale)
{
    // reference: clamp<int8_t>(float_sum / scale_factor), truncating cast
    const float v = (float)sum / scale;
    return (int8_t)fmaxf(-128.0f, fminf(127.0f, v));
}

constexpr int kPfRows = 64;  // stage rows up to which the next channel is prefetched in registers

// Input word (t, f, w) lives at t * stride_t + f * stride_f + w: TFB
// (stride_t = F * nwords, stride_f = nwords) or channel-major FTB
// (stride_t = nwords, stride_f = T * nwords), which keeps a channel's rows
// together.  PF: the next channel's stage (<= kPfRows rows) is loaded into
// registers while the current one is summed.
template <int DPW, int TT, bool WIDE, bool PF>
__global__ void __launch_bounds__(256)
idisp_kernel(const uint32_t* __restrict__ tfb, uint32_t* __restrict__ tdb,
             const int* __restrict__ delays, const int2* __restrict__ span,
             const int2* __restrict__ tiles, int nchans, int nwords, int ndms, int ts,
             int max_delay, long nsamples, int nout, int tb0, float scale, long stride_t, long stride_f)
{
    extern __shared__ uint4 stage[];  // [rows][16] uint4 = [rows][64] words
    const uint32_t* rows = reinterpret_cast<const uint32_t*>(stage);
    const int tile  = blockIdx.x;
    const int chunk = blockIdx.y;
    const int tb    = tb0 + blockIdx.z;
    const int wave  = threadIdx.x >> 6;
    const int lane  = threadIdx.x & 63;
    const int2 td   = tiles[tile];
    const int t0    = tb * TT;
    const long in0  = (long)max_delay + (long)t0 * ts;

    uint32_t e[DPW][TT], o[DPW][TT];
    uint32_t w32[WIDE ? DPW : 1][WIDE ? TT : 1][4];
#pragma unroll
    for(int j = 0; j < DPW; ++j)
#pragma unroll
        for(int i = 0; i < TT; ++i) {
            e[j][i] = 0;
            o[j][i] = 0;
            if constexpr(WIDE) {
#pragma unroll
                for(int k = 0; k < 4; ++k) w32[j][i][k] = 0;
            }
        }
    int pending = 0;  // biased bytes in the 16-bit lanes (WIDE only)

    // 16-byte pieces of channel f's stage (rows 16-byte aligned: nwords % 4 == 0)
    auto piece = [&](int f, long lo, int i) {
        const int r = i >> 4, q = i & 15;
        const int w4 = chunk * 64 + q * 4;
        uint4 v = make_uint4(0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u);
        if(w4 < nwords && lo + r < nsamples) {
            v = *reinterpret_cast<const uint4*>(tfb + (lo + r) * stride_t + f * stride_f + w4);
            v.x ^= 0x80808080u;
            v.y ^= 0x80808080u;
            v.z ^= 0x80808080u;
            v.w ^= 0x80808080u;
        }
        return v;
    };
    constexpr int NPF = PF ? kPfRows * 16 / 256 : 1;
    uint4 pre[NPF];
    if constexpr(PF) {
        const int2 sp = span[(size_t)tile * nchans];
        const int nr = TT * ts + sp.y - sp.x;
#pragma unroll
        for(int k = 0; k < NPF; ++k) {
            const int i = threadIdx.x + 256 * k;
            if(i < nr * 16) pre[k] = piece(0, in0 - sp.y, i);
        }
    }

    for(int f = 0; f < nchans; ++f) {
        const int2 sp   = span[(size_t)tile * nchans + f];
        const long lo   = in0 - sp.y;
        const int nrows = TT * ts + sp.y - sp.x;
        __syncthreads();
        if constexpr(PF) {
#pragma unroll
            for(int k = 0; k < NPF; ++k) {
                const int i = threadIdx.x + 256 * k;
                if(i < nrows * 16) stage[i] = pre[k];
            }
            if(f + 1 < nchans) {  // next channel's rows, in flight during the sums
                const int2 sn = span[(size_t)tile * nchans + f + 1];
                const int nr = TT * ts + sn.y - sn.x;
#pragma unroll
                for(int k = 0; k < NPF; ++k) {
                    const int i = threadIdx.x + 256 * k;
                    if(i < nr * 16) pre[k] = piece(f + 1, in0 - sn.y, i);
                }
            }
        } else if((nwords & 3) == 0) {
            for(int i = threadIdx.x; i < nrows * 16; i += 256) stage[i] = piece(f, lo, i);
        } else {
            uint32_t* st32 = reinterpret_cast<uint32_t*>(stage);
            for(int i = threadIdx.x; i < nrows * 64; i += 256) {
                const int r = i >> 6, q = i & 63;
                const int w = chunk * 64 + q;
                uint32_t v = 0x80808080u;
                if(w < nwords && lo + r < nsamples) v = tfb[(lo + r) * stride_t + f * stride_f + w] ^ 0x80808080u;
                st32[i] = v;
            }
        }
        __syncthreads();
#pragma unroll
        for(int j = 0; j < DPW; ++j) {
            const int dl = wave + 4 * j;
            if(dl < td.y) {
                const int delta = delays[(size_t)(td.x + dl) * nchans + f];
                const uint32_t* src = rows + (sp.y - delta) * 64 + lane;
#pragma unroll
                for(int i = 0; i < TT; ++i)
                    for(int s = 0; s < ts; ++s) id_add(src[(i * ts + s) * 64], e[j][i], o[j][i]);
            }
        }
        if constexpr(WIDE) {
            pending += ts;
            if(pending + ts > 256 || f == nchans - 1) {
#pragma unroll
                for(int j = 0; j < DPW; ++j)
#pragma unroll
                    for(int i = 0; i < TT; ++i) {
                        w32[j][i][0] += e[j][i] & 0xFFFFu;
                        w32[j][i][1] += o[j][i] & 0xFFFFu;
                        w32[j][i][2] += e[j][i] >> 16;
                        w32[j][i][3] += o[j][i] >> 16;
                        e[j][i] = 0;
                        o[j][i] = 0;
                    }
                pending = 0;
            }
        }
    }

    const int word = chunk * 64 + lane;
    if(word >= nwords) return;
    const int32_t bias = 128 * nchans * ts;
#pragma unroll
    for(int j = 0; j < DPW; ++j) {
        const int dl = wave + 4 * j;
        if(dl >= td.y) continue;
#pragma unroll
        for(int i = 0; i < TT; ++i) {
            if(t0 + i >= nout) continue;
            int32_t s[4];
            if constexpr(WIDE) {
#pragma unroll
                for(int k = 0; k < 4; ++k) s[k] = (int32_t)w32[j][i][k] - bias;
            } else {
                s[0] = (int32_t)(e[j][i] & 0xFFFFu) - bias;
                s[1] = (int32_t)(o[j][i] & 0xFFFFu) - bias;
                s[2] = (int32_t)(e[j][i] >> 16) - bias;
                s[3] = (int32_t)(o[j][i] >> 16) - bias;
            }
            const uint32_t packed = (uint32_t)(uint8_t)id_quant(s[0], scale) |
                                    ((uint32_t)(uint8_t)id_quant(s[1], scale) << 8) |
                                    ((uint32_t)(uint8_t)id_quant(s[2], scale) << 16) |
                                    ((uint32_t)(uint8_t)id_quant(s[3], scale) << 24);
            tdb[((size_t)(t0 + i) * ndms + td.x + dl) * nwords + word] = packed;
        }
    }
}

constexpr int kRowsCap = 256;  // staged rows per channel: 64 KB of LDS

// ---------------------------------------------------------------- MFMA form

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMfRows  = 128;   // staged rows per channel, 16 waves (one DM each) per workgroup
constexpr int kMfWaves = 16;
constexpr int kSmRows  = 64;    // the same where 8 DMs' rows are few: 8 waves, two workgroups per CU
constexpr int kSmWaves = 8;
constexpr int kMfTabCh = 512;   // channels whose delay tables are held in LDS at a time
constexpr int kMfMaxTs = 8;

// Rows that a channel's stage of `rcap` rows holds at tscrunch ts (a whole
// number of rows per phase of ts).
constexpr int id_stage_rows(int rcap, int ts) { return rcap / ts * ts; }

// Work items are dealt to the 8 XCDs in contiguous runs, and a run is walked
// in groups of kIdTbGroup time blocks x kIdTileGroup DM tiles of one chunk:
// the 32 workgroups that one XCD runs together read overlapping rows (next
// time blocks; DM tiles of neighbouring delays), which its L2 then serves.
constexpr int kIdTbGroup = 8, kIdTileGroup = 4;

struct IdArgs {
    const int8_t* in;
    int8_t* tdb;
    const uint8_t* rel;  // [tile][channel][NW]: the tile's largest delay in the channel less the DM's
    const int2* span;    // [tile][channel]: the tile's smallest and largest delay
    const int2* tiles;   // [tile]: first DM, DMs
    int ntiles, chunk0, nchunks, ntb;
    long w0, nwork;
    int nchans, W, ndms, max_delay;
    long nsamples;
    int nout;
    float scale;
    long stride_t, stride_f;  // bytes
};

// A workgroup of NW waves owns 16 NTT output samples, 128 bytes of beams (a
// chunk) and a tile of up to NW consecutive DMs, one per wave.  Per quad of
// channels the union of the rows its DMs read, [in0 - max delay, in0 +
// 16 NTT TS - min delay) per channel, goes from global memory straight into
// one of two LDS stage buffers (global_load_lds_dwordx4: lane L of a wave's
// load writes the 16-byte slot L of a 1 KB block, eight rows) while the
// previous quad's products read the other, one barrier per quad.  Input byte
// (t, f, b) lives at t * stride_t + f * stride_f + b (TFB or FTB).  NBG: 16-beam
// groups of the chunk (4 where only 64 bytes of it hold beams).
//
// Stage layout: rows of 128 bytes.  Logical row r lies at row (r mod TS) RP +
// r / TS, so that the 16 rows TS apart that one read takes are neighbours,
// and 16-byte piece c of stored row r' in slot c ^ ((r' / 2) mod 8): any 16
// consecutive rows then start on distinct banks.  (Rows TS apart put a read
// on 16 / TS banks: 300 DMs x 404 beams x 64 channels x 3000 samples at
// tscrunch 4 took 5.4 ms.)  That holds for the rows of one channel: a read
// takes those of four, each from its own first row, and what these lose to
// each other is left (24 % of the LDS's active cycles at tscrunch 1, 10 % at
// 4).
//
// What bounds it: the round trip of a quad's row loads, issued after the
// barrier that frees their buffer.  1024 DMs x 512 beams x 256 channels x 4096
// samples take 9.9 to 10.4 ms by card (5.3e13 to 5.6e13 sums/s), 6.6 ms
// without the loads, 8.4 ms without the products; of 2.3e7 cycles a CU's LDS
// is active for 52 %, 5.75 cycles per read of a product (1.4 of them the
// conflicts above), the matrix cores for 37 %.  A load therefore costs no address
// arithmetic: per channel a table in LDS, filled once per kMfTabCh channels,
// holds where its rows begin and end, a buffer resource over them takes the
// lane's fixed offset and its range check stands for the row tests, and a
// wave loads rows of one channel only.  (With 64-bit addresses and the tests
// formed per load, and the delays loaded per quad, the VALU was busy with
// them for two thirds of the time: 13.5 ms.  Touching the rows of the quad
// after the next ahead of time, 16.5 ms with that form.)
//
// Slots past the tile's rows or the input are zero or keep stale bytes, those
// past W keep stale bytes, and a row's last piece may hold the next row's
// first bytes: no stored output reads them (rows past the span are read by no
// DM of the tile, rows past the input feed only output samples >= nout, beams
// past W only beams >= W, and the one-hot products sum each beam from its own
// bytes).
template <int NW, int NTT, int NBG, int RCAP, int TS, bool BIG>
__device__ __forceinline__ void idisp_tile(const IdArgs& p)
{
    constexpr int TT  = 16 * NTT;
    constexpr int RP  = RCAP / TS;       // stored rows per phase
    constexpr int QB  = 4 * RCAP * 128;
    static_assert(RCAP == 8 * NW, "a wave loads eight rows (1 KB) of each channel of a quad");
    // two arrays, not one: the compiler then knows that a buffer's reads do
    // not touch the loads in flight into the other (with one array it waits
    // for every row load before any read)
    __shared__ __attribute__((aligned(16))) int8_t stage0[QB];
    __shared__ __attribute__((aligned(16))) int8_t stage1[QB];
    __shared__ __attribute__((aligned(16))) int4 tab[kMfTabCh];  // offset of the first row (64 bits), bytes (BIG: see below), rows
    __shared__ __attribute__((aligned(16))) uint8_t tab_rel[kMfTabCh * NW];  // [channel][wave]: rows to the DM's first

    const long per = (p.nwork + 7) / 8;
    const long wl  = (long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if(wl >= p.nwork) return;  // whole workgroup, before any barrier
    const long w = p.w0 + wl;
    constexpr int GRP = kIdTbGroup * kIdTileGroup;
    const int gi = (int)(w % GRP);
    const long rest  = w / GRP;
    const int chunk  = p.chunk0 + (int)(rest % p.nchunks);
    const long blk   = rest / p.nchunks;
    const int ntbb   = (p.ntb + kIdTbGroup - 1) / kIdTbGroup;
    const int tb     = (int)(blk % ntbb) * kIdTbGroup + gi % kIdTbGroup;
    const int tile   = (int)(blk / ntbb) * kIdTileGroup + gi / kIdTbGroup;
    if(tb >= p.ntb || tile >= p.ntiles) return;  // whole workgroup, before any barrier
    const int2 td    = p.tiles[tile];
    const int t0     = tb * TT;
    const long in0   = (long)p.max_delay + (long)t0 * TS;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, g = lane >> 4;
    const int b0 = chunk * 128;
    const bool active = wv < td.y;        // this wave's DM is in the tile
    const bool ragged = (p.W & 15) != 0;  // a row's last piece may pass the input's end

    // Staging: wave w loads 8-row blocks w mod WPC + WPC k (k < 4) of channel
    // w / WPC of every quad, so a quad costs a wave one table entry.  A lane's
    // offsets within a channel's rows are the same for all quads.
    constexpr int WPC = NW / 4;
    const int sc = wv / WPC;  // the wave's channel of a quad
    auto stored_row = [&](int k) { return (wv % WPC + WPC * k) * 8 + (lane >> 3); };
    auto piece = [&](int rs) { return b0 + (((lane & 7) ^ ((rs >> 1) & 7)) << 4); };
    uint32_t voff[4];
#pragma unroll
    for(int k = 0; k < 4; ++k) {
        const int rs = stored_row(k), b = piece(rs);
        const bool in = rs < RP * TS && b < p.W;
        voff[k] = in ? (uint32_t)(rs % RP * TS + rs / RP) * (uint32_t)p.stride_t + b : 0xFFFFFFF0u;
    }
    // quad q's rows into stg: through a buffer resource that ends with the
    // channel's last row (a load past it stores zeros), or where 32 bits do
    // not span the stage's rows (BIG) by 64-bit addresses
    auto issue = [&](int f0, int q, int8_t* stg) {
        const int4 e = tab[4 * q + sc];
        const unsigned lo = __builtin_amdgcn_readfirstlane(e.x), hi = __builtin_amdgcn_readfirstlane(e.y);
        const int nr = __builtin_amdgcn_readfirstlane(e.w);
        const int8_t* src = p.in + ((unsigned long)hi << 32 | lo);
        if constexpr(BIG) {
            const bool last = __builtin_amdgcn_readfirstlane(e.z) != 0;  // the last row ends the input
#pragma unroll
            for(int k = 0; k < 4; ++k) {
                const int rs = stored_row(k), b = piece(rs), r = rs % RP * TS + rs / RP;
                const bool end = last && r == nr - 1;
                if(rs < RP * TS && r < nr && (end ? b + 16 <= p.W : b < p.W))
                    __builtin_amdgcn_global_load_lds(
                        src + (unsigned long)r * p.stride_t + b,
                        (__attribute__((address_space(3))) void*)(stg + (sc * RCAP + (wv % WPC + WPC * k) * 8) * 128),
                        16, 0, 0);
            }
        } else {
            const auto rs = buffer_rsrc(src, __builtin_amdgcn_readfirstlane(e.z));
#pragma unroll
            for(int k = 0; k < 4; ++k)
                if(TS > 1 || (wv % WPC + WPC * k) * 8 < nr)  // uniform
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        rs, (__attribute__((address_space(3))) void*)(stg + (sc * RCAP + (wv % WPC + WPC * k) * 8) * 128),
                        16, voff[k], 0, 0, 0);
        }
    };
    // the last piece of the input's last row (the last channel's), W mod 16
    // bytes, by words: a whole piece would pass the input's end.  Called once
    // the wave's loads have arrived, by the wave that loaded the row (its load
    // of the slot stored zeros).
    auto finish = [&](int f0, int q, int8_t* stg) {
        if(!ragged || f0 + 4 * q + 4 < p.nchans || p.W - b0 > 128) return;  // wave-uniform
        const int r = tab[4 * q + 3].w - 1;
        const int rs = r % TS * RP + r / TS, c = (p.W - b0) >> 4;
        if(in0 - p.span[(size_t)tile * p.nchans + p.nchans - 1].y + r != p.nsamples - 1 ||
           wv != 3 * WPC + rs / 8 % WPC || lane >= (p.W & 15) / 4)
            return;
        *reinterpret_cast<uint32_t*>(stg + (3 * RCAP + rs) * 128 + ((c ^ ((rs >> 1) & 7)) << 4) + 4 * lane) =
            *reinterpret_cast<const uint32_t*>(p.in + (p.nsamples - 1) * p.stride_t +
                                               (long)(p.nchans - 1) * p.stride_f + b0 + 16 * c + 4 * lane);
    };

    v4i sel = {0, 0, 0, 0};
    sel[n >> 2] = 1 << (8 * (n & 3));
    v4i acc[NTT][NBG];
#pragma unroll
    for(int tt = 0; tt < NTT; ++tt)
#pragma unroll
        for(int bg = 0; bg < NBG; ++bg) acc[tt][bg] = v4i{0, 0, 0, 0};

    auto products = [&](int q, const int8_t* stg) {
        if(!active) return;  // wave-uniform
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int n = ln & 15, g = ln >> 4;
        const int rel = tab_rel[(4 * q + g) * NW + wv];
#pragma unroll
        for(int s = 0; s < TS; ++s) {
            const int k = rel + s;
            const int rs = k % TS * RP + k / TS + n;
            const int base = (g * RCAP + rs) * 128 + (((rs >> 1) & 7) << 4);
#pragma unroll
            for(int tt = 0; tt < NTT; ++tt) {
                v4i bv[NBG];  // the row's reads in flight together
#pragma unroll
                for(int bg = 0; bg < NBG; ++bg)
                    bv[bg] = *reinterpret_cast<const v4i*>(stg + (base ^ (bg << 4)) + tt * 2048);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for(int bg = 0; bg < NBG; ++bg)
                    acc[tt][bg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(sel, bv[bg], acc[tt][bg], 0, 0, 0);
            }
        }
    };
    // quad q's rows are in stg, and every wave is done with the other buffer
    auto settle = [&](int f0, int q, int8_t* stg) {
        __builtin_amdgcn_s_waitcnt(0);
        finish(f0, q, stg);
        __syncthreads();
    };

    for(int f0 = 0; f0 < p.nchans; f0 += kMfTabCh) {
        const int nf = min(kMfTabCh, p.nchans - f0), nq = nf / 4;
        // workgroups that run together on an XCD take each eight quads in
        // rotated order (the sums are exact in any): their row loads then
        // fall on different channels' lines
        auto order = [&](int q) { return (q | 7) < nq ? (q & ~7) | ((q + (int)wl) & 7) : q; };
        __syncthreads();  // the last range's products are done
        for(int i = threadIdx.x; i < nf; i += NW * 64) {
            const int2 sp = p.span[(size_t)tile * p.nchans + f0 + i];
            const long lo = in0 - sp.y, at = lo * p.stride_t + (f0 + i) * p.stride_f;
            const int nr = (int)min((long)(TT * TS + sp.y - sp.x), p.nsamples - lo);
            // the input's very last piece, where it is no whole one, is finish()'s
            const bool end = ragged && f0 + i == p.nchans - 1 && lo + nr == p.nsamples;
            // BIG has no use for the bytes: whether finish() loads that piece stands there
            const long bytes = (nr - 1) * p.stride_t + (end ? p.W & ~15 : p.W);
            tab[i] = make_int4((int)at, (int)(at >> 32), BIG ? (int)end : (int)bytes, nr);
            using R = typename std::conditional<NW == 16, uint4, uint2>::type;
            reinterpret_cast<R*>(tab_rel)[i] =
                reinterpret_cast<const R*>(p.rel)[(size_t)tile * p.nchans + f0 + i];
        }
        __syncthreads();
        // quads alternate between the buffers: even positions in stage0, odd in stage1
        issue(f0, order(0), stage0);
        for(int q = 0; q < nq; q += 2) {
            settle(f0, order(q), stage0);
            if(q + 1 < nq) issue(f0, order(q + 1), stage1);
            products(order(q), stage0);
            if(q + 1 < nq) {
                settle(f0, order(q + 1), stage1);
                if(q + 2 < nq) issue(f0, order(q + 2), stage0);
                products(order(q + 1), stage1);
            }
        }
    }

    // C lane (n, g), register r: beam b0 + 16 bg + 4 g + r at sample t0 + 16 tt + n
    if(!active) return;
#pragma unroll
    for(int tt = 0; tt < NTT; ++tt) {
        const int t = t0 + 16 * tt + n;
        if(t >= p.nout) continue;
        int8_t* o = p.tdb + ((size_t)t * p.ndms + td.x + wv) * p.W;
#pragma unroll
        for(int bg = 0; bg < NBG; ++bg) {
            const int b = b0 + 16 * bg + 4 * g;
            if(b >= p.W) continue;
            const v4i a = acc[tt][bg];
            const uint32_t packed = (uint32_t)(uint8_t)id_quant(a[0], p.scale) |
                                    ((uint32_t)(uint8_t)id_quant(a[1], p.scale) << 8) |
                                    ((uint32_t)(uint8_t)id_quant(a[2], p.scale) << 16) |
                                    ((uint32_t)(uint8_t)id_quant(a[3], p.scale) << 24);
            *reinterpret_cast<uint32_t*>(o + b) = packed;
        }
    }
}

// 32 output samples per workgroup
template <int NW, int NBG, int RCAP, int TS, bool BIG>
__global__ void __launch_bounds__(NW * 64, 4) idisp_dma_kernel(IdArgs p)
{
    idisp_tile<NW, 2, NBG, RCAP, TS, BIG>(p);
}

// 16 output samples per workgroup: tscrunch above 2, where 32 samples' rows
// would leave the stage no room for the DMs' delays
template <int NBG, int TS, bool BIG>
__global__ void __launch_bounds__(kMfWaves * 64, 4) idisp_mfma_kernel(IdArgs p)
{
    idisp_tile<kMfWaves, 1, NBG, kMfRows, TS, BIG>(p);
}

template <int NBG, bool BIG>
int idisp_launch_mfma(int ts, bool small, const IdArgs& a, hipStream_t st)
{
    const dim3 grid((unsigned)(8 * ((a.nwork + 7) / 8))), block(64 * (small ? kSmWaves : kMfWaves));
    switch(small ? 0 : ts) {
#define SW_IDM(TS, ...) \
    case TS: hipLaunchKernelGGL((__VA_ARGS__), grid, block, 0, st, a); break;
        SW_IDM(0, idisp_dma_kernel<kSmWaves, NBG, kSmRows, 1, BIG>)
        SW_IDM(1, idisp_dma_kernel<kMfWaves, NBG, kMfRows, 1, BIG>)
        SW_IDM(2, idisp_dma_kernel<kMfWaves, NBG, kMfRows, 2, BIG>)
        SW_IDM(3, idisp_mfma_kernel<NBG, 3, BIG>)
        SW_IDM(4, idisp_mfma_kernel<NBG, 4, BIG>)
        SW_IDM(5, idisp_mfma_kernel<NBG, 5, BIG>)
        SW_IDM(6, idisp_mfma_kernel<NBG, 6, BIG>)
        SW_IDM(7, idisp_mfma_kernel<NBG, 7, BIG>)
        SW_IDM(8, idisp_mfma_kernel<NBG, 8, BIG>)
#undef SW_IDM
    }
    SW_LAUNCH_CHECK();
    return SW_OK;
}

void free_plan_device(sw_idisp* p)
{
    (void)hipFree(p->d_delays);
    (void)hipFree(p->d_rel);
    (void)hipFree(p->d_span);
    (void)hipFree(p->d_tiles);
    p->d_delays = nullptr;
    p->d_rel = nullptr;
    p->d_span = nullptr;
    p->d_tiles = nullptr;
}

} // namespace
} // namespace sw

extern "C" int sw_id_delays(const float* dms, int ndms, const double* chan_freqs, int nchans,
                            double tsamp, int* h_delays, int* max_delay)
{
    SW_CHECK_ARG(dms && chan_freqs && h_delays && ndms > 0 && nchans > 0 && tsamp > 0, "bad argument");
    // DMSampleDelay(dm, f_ref = channel_frequencies().front(), tsamp)(f)
    const double f_ref = chan_freqs[0];
    int mx = 0;
    for(int d = 0; d < ndms; ++d)
        for(int c = 0; c < nchans; ++c) {
            const double f = chan_freqs[c];
            const double delay = sw::kDmConstHzS * (1 / (f_ref * f_ref) - 1 / (f * f)) * (double)dms[d];
            const int v = (int)(delay / tsamp + 0.5);
            h_delays[(size_t)d * nchans + c] = v;
            mx = std::max(mx, v);
        }
    if(max_delay) *max_delay = mx;
    return SW_OK;
}

extern "C" int sw_channel_frequencies(double centre_frequency, double bandwidth, int nchans,
                                      double* h_freqs)
{
    // PipelineConfig::calculate_channel_frequencies,
    // cpp/skyweaver/src/PipelineConfig.cpp:188-203
    SW_CHECK_ARG(h_freqs && nchans > 0, "bad argument");
    const double chbw = bandwidth / nchans;
    const double fbottom = centre_frequency - bandwidth / 2.0;
    for(int c = 0; c < nchans; ++c) h_freqs[c] = fbottom + chbw / 2.0 + (chbw * c);
    return SW_OK;
}

extern "C" int sw_ddplan_parse_block(const char* spec, float* coherent_dm, int* tscrunch,
                                     float* h_dms, int max_dms, int* ndms)
{
    // DedispersionPlan::add_block(std::string), cpp/skyweaver/src/DedispersionPlan.cpp:17-78:
    // "cdm", "cdm:tscrunch" or "cdm:begin:end:step:tscrunch"; the incoherent
    // DMs of the last form are accumulated in float (dm += step while dm < end),
    // and an empty range yields {begin}.
    SW_CHECK_ARG(spec && coherent_dm && tscrunch && ndms, "null argument");
    std::vector<std::string> parts;
    {
        std::stringstream ss(spec);
        std::string item;
        while(std::getline(ss, item, ':')) parts.push_back(item);
    }
    std::vector<float> dms;
    try {
        if(parts.size() == 1 || parts.size() == 2) {
            *coherent_dm = std::stof(parts[0]);
            *tscrunch = parts.size() == 2 ? std::stoi(parts[1]) : 1;
            dms.push_back(*coherent_dm);
        } else if(parts.size() == 5) {
            *coherent_dm = std::stof(parts[0]);
            const float b = std::stof(parts[1]), e = std::stof(parts[2]), st = std::stof(parts[3]);
            *tscrunch = std::stoi(parts[4]);
            for(float dm = b; dm < e; dm += st) {
                dms.push_back(dm);
                if(dms.size() > (size_t)1 << 24) break;
            }
            if(dms.empty()) dms.push_back(b);
        } else {
            sw::set_error(std::string("Block defition string of unexpected size: ") + spec);
            return SW_ERR_INVALID;
        }
    } catch(std::invalid_argument& e) {
        sw::set_error(std::string("Error parsing block definition string: ") + e.what());
        return SW_ERR_INVALID;
    } catch(std::out_of_range&) {
        sw::set_error("Block definition value out of range");
        return SW_ERR_INVALID;
    }
    *ndms = (int)dms.size();
    if(h_dms) {
        SW_CHECK_ARG(max_dms >= (int)dms.size(), "DM buffer too small");
        std::memcpy(h_dms, dms.data(), sizeof(float) * dms.size());
    }
    return SW_OK;
}

extern "C" int sw_idisp_create(const sw_idisp_config* cfg, sw_idisp** out)
{
    SW_CHECK_ARG(cfg && out, "null argument");
    *out = nullptr;
    SW_CHECK_ARG(cfg->nchans > 0 && cfg->ndms > 0 && cfg->dms, "empty plan");
    SW_CHECK_ARG(cfg->tscrunch > 0 && cfg->cb_tscrunch > 0, "tscrunch must be positive");
    SW_CHECK_ARG(cfg->bandwidth != 0.0, "bandwidth must be non-zero");
    auto p = std::make_unique<sw_idisp>();
    p->nchans = cfg->nchans;
    p->ndms = cfg->ndms;
    p->tscrunch = cfg->tscrunch;
    p->dms.assign(cfg->dms, cfg->dms + cfg->ndms);
    std::vector<double> freqs(cfg->nchans);
    if(cfg->chan_freqs)
        freqs.assign(cfg->chan_freqs, cfg->chan_freqs + cfg->nchans);
    else
        sw_channel_frequencies(cfg->centre_frequency, cfg->bandwidth, cfg->nchans, freqs.data());
    const double chbw = cfg->bandwidth / cfg->nchans;
    const double tsamp = cfg->cb_tscrunch / chbw;
    p->delays.resize((size_t)cfg->ndms * cfg->nchans);
    sw_id_delays(p->dms.data(), p->ndms, freqs.data(), p->nchans, tsamp, p->delays.data(), &p->max_delay);
    for(int v: p->delays)
        SW_CHECK_ARG(v >= 0, "channel frequencies must not lie below the first channel's");
    p->scale = (float)std::sqrt((double)((size_t)p->nchans * p->tscrunch));

    // tiling: TT output samples per workgroup, tiles of consecutive DMs whose
    // union of read rows fits the LDS stage
    const int F = p->nchans;
    std::vector<int2> span;
    auto tile_dms = [&](int cap, int dmax_tile) {
        p->tiles.clear();
        span.clear();
        p->rows_cap = 0;
        for(int d = 0; d < p->ndms;) {
            int n = 1;
            while(n < dmax_tile && d + n < p->ndms) {
                int worst = 0;
                for(int f = 0; f < F; ++f) {
                    int lo = INT32_MAX, hi = INT32_MIN;
                    for(int k = 0; k <= n; ++k) {
                        lo = std::min(lo, p->delays[(size_t)(d + k) * F + f]);
                        hi = std::max(hi, p->delays[(size_t)(d + k) * F + f]);
                    }
                    worst = std::max(worst, hi - lo);
                }
                if(worst + p->tt * p->tscrunch > cap) break;
                ++n;
            }
            p->tiles.push_back(make_int2(d, n));
            int rows = 0;
            for(int f = 0; f < F; ++f) {
                int lo = INT32_MAX, hi = INT32_MIN;
                for(int k = 0; k < n; ++k) {
                    lo = std::min(lo, p->delays[(size_t)(d + k) * F + f]);
                    hi = std::max(hi, p->delays[(size_t)(d + k) * F + f]);
                }
                span.push_back(make_int2(lo, hi));
                rows = std::max(rows, hi - lo + p->tt * p->tscrunch);
            }
            p->rows_cap = std::max(p->rows_cap, rows);
            d += n;
        }
    };
    std::vector<uint8_t> rel;
    p->mfma = cfg->kernel == 0 && p->nchans % 4 == 0 && 16 * p->tscrunch <= sw::kMfRows;
    if(p->mfma) {
        static_assert(16 * sw::kMfMaxTs <= sw::kMfRows && 16 * (sw::kMfMaxTs + 1) > sw::kMfRows, "every tscrunch has a kernel");
        // 32 output samples per workgroup while that leaves half of the stage
        // for the DMs' delays, else 16
        p->tt = 32 * p->tscrunch <= sw::kMfRows / 2 ? 32 : 16;
        // where every run of 8 DMs fits the small stage, two workgroups of 8
        // waves share a CU and one's products cover the other's waits;
        // otherwise 16 DMs share the staged rows
        if(p->tscrunch == 1) {
            tile_dms(sw::kSmRows, sw::kSmWaves);
            p->small = (int)p->tiles.size() == (p->ndms + sw::kSmWaves - 1) / sw::kSmWaves;
        }
        if(!p->small) tile_dms(sw::id_stage_rows(sw::kMfRows, p->tscrunch), sw::kMfWaves);
        const int nw = p->small ? sw::kSmWaves : sw::kMfWaves;
        rel.assign(p->tiles.size() * F * nw, 0);
        for(size_t t = 0; t < p->tiles.size(); ++t)
            for(int f = 0; f < F; ++f)
                for(int k = 0; k < p->tiles[t].y; ++k)
                    rel[(t * F + f) * nw + k] =
                        (uint8_t)(span[t * F + f].y - p->delays[(size_t)(p->tiles[t].x + k) * F + f]);
    } else {
        p->wide = (long)p->nchans * p->tscrunch > 256;
        p->tt = p->wide ? 8 : 16;
        if(p->tt * p->tscrunch > sw::kRowsCap / 2) p->tt = 4;
        if(p->tt * p->tscrunch > sw::kRowsCap) {
            sw::set_error("incoherent dedispersion tscrunch too large (at most 64)");
            return SW_ERR_UNSUPPORTED;
        }
        p->dpw = 2;
        tile_dms(sw::kRowsCap, 8);
    }
    if(!rel.empty()) {
        SW_HIP_TRY(hipMalloc(&p->d_rel, rel.size()));
        SW_HIP_TRY(hipMemcpy(p->d_rel, rel.data(), rel.size(), hipMemcpyHostToDevice));
    }
    SW_HIP_TRY(hipMalloc(&p->d_delays, sizeof(int) * p->delays.size()));
    SW_HIP_TRY(hipMalloc(&p->d_span, sizeof(int2) * span.size()));
    SW_HIP_TRY(hipMalloc(&p->d_tiles, sizeof(int2) * p->tiles.size()));
    SW_HIP_TRY(hipMemcpy(p->d_delays, p->delays.data(), sizeof(int) * p->delays.size(), hipMemcpyHostToDevice));
    SW_HIP_TRY(hipMemcpy(p->d_span, span.data(), sizeof(int2) * span.size(), hipMemcpyHostToDevice));
    SW_HIP_TRY(hipMemcpy(p->d_tiles, p->tiles.data(), sizeof(int2) * p->tiles.size(), hipMemcpyHostToDevice));
    *out = p.release();
    return SW_OK;
}

extern "C" int sw_idisp_destroy(sw_idisp* p)
{
    if(p) {
        sw::free_plan_device(p);
        delete p;
    }
    return SW_OK;
}

extern "C" const char* sw_idisp_kernel(const sw_idisp* p)
{
    if(!p) return "";
    if(!p->mfma) return "idisp_kernel";
    return p->tt == 32 ? "idisp_dma_kernel" : "idisp_mfma_kernel";
}

extern "C" int sw_idisp_info(const sw_idisp* p, int* max_delay, int* h_delays, float* scale)
{
    SW_CHECK_ARG(p, "null plan");
    if(max_delay) *max_delay = p->max_delay;
    if(h_delays) std::memcpy(h_delays, p->delays.data(), sizeof(int) * p->delays.size());
    if(scale) *scale = p->scale;
    return SW_OK;
}

namespace sw {
int idisp_launch(sw_idisp* p, const void* d_in, size_t nsamples, int nbeams, int nvec, void* d_tdb, bool ftb,
                 hipStream_t st);
}

extern "C" int sw_idisp_dedisperse(sw_idisp* p, const void* d_tfb, size_t nsamples, int nbeams, int nvec,
                                   void* d_tdb, void* stream)
{
    return sw::idisp_launch(p, d_tfb, nsamples, nbeams, nvec, d_tdb, false, sw::as_stream(stream));
}

extern "C" int sw_idisp_dedisperse_ftb(sw_idisp* p, const void* d_ftb, size_t nsamples, int nbeams, int nvec,
                                       void* d_tdb, void* stream)
{
    return sw::idisp_launch(p, d_ftb, nsamples, nbeams, nvec, d_tdb, true, sw::as_stream(stream));
}

int sw::idisp_launch(sw_idisp* p, const void* d_tfb, size_t nsamples, int nbeams, int nvec, void* d_tdb, bool ftb,
                     hipStream_t st)
{
    SW_CHECK_ARG(p && d_tfb && d_tdb, "null argument");
    SW_CHECK_ARG(nbeams > 0 && (nvec == 1 || nvec == 4), "nvec must be 1 (int8) or 4 (char4)");
    if(nsamples <= (size_t)p->max_delay) {
        sw::set_error("Fewer than max_sample_delay samples passed to dedisperse method");
        return SW_ERR_INVALID;
    }
    if((nsamples - p->max_delay) % p->tscrunch != 0) {
        sw::set_error("(nsamples - max_sample_delay) must be a multiple of tscrunch;");
        return SW_ERR_INVALID;
    }
    const long nbv = (long)nbeams * nvec;
    SW_CHECK_ARG(nbv % 4 == 0, "nbeams * nvec must be a multiple of 4");
    SW_CHECK_ARG(((uintptr_t)d_tfb & 15) == 0 && ((uintptr_t)d_tdb & 3) == 0, "misaligned buffer");
    const int nwords = (int)(nbv / 4);
    const int nout = (int)((nsamples - p->max_delay) / p->tscrunch);
    const int nchunks = (nwords + 63) / 64;
    const int ntb = (nout + p->tt - 1) / p->tt;
    const size_t lds = (size_t)p->rows_cap * 256;
    const long stride_t = ftb ? nwords : (long)p->nchans * nwords;
    const long stride_f = ftb ? (long)nsamples * nwords : nwords;
    if(p->mfma) {
        // chunks of 128 bytes of beams; a last one of at most 64 by itself,
        // with half of the products.  big: 32 bits do not span a stage's rows
        const bool big = 128 * stride_t * 4 + nbv >= 0xFFFFFFF0L;
        const int last = (int)(nbv % 128), nfull = (int)(nbv / 128) + (last > 64 || (big && last > 0));
        const long ntiles = (long)p->tiles.size();
        for(int half = 0; half < 2; ++half) {
            const int chunk0 = half ? nfull : 0, nchunks128 = half ? (last > 0 && last <= 64 && !big) : nfull;
            const long nwork = (ntiles + sw::kIdTileGroup - 1) / sw::kIdTileGroup * sw::kIdTileGroup * nchunks128 *
                               (((long)ntb + sw::kIdTbGroup - 1) / sw::kIdTbGroup * sw::kIdTbGroup);
            const long max_launch = 2L << 20;  // work items per launch (grid x 1024 threads < 2^32)
            for(long w0 = 0; w0 < nwork; w0 += max_launch) {
                const sw::IdArgs a{static_cast<const int8_t*>(d_tfb), static_cast<int8_t*>(d_tdb), p->d_rel,
                                   p->d_span, p->d_tiles, (int)ntiles, chunk0, nchunks128, ntb, w0,
                                   std::min(max_launch, nwork - w0), p->nchans, (int)nbv, p->ndms, p->max_delay,
                                   (long)nsamples, nout, p->scale, stride_t * 4, stride_f * 4};
                const int rc = half  ? sw::idisp_launch_mfma<4, false>(p->tscrunch, p->small, a, st)
                               : big ? sw::idisp_launch_mfma<8, true>(p->tscrunch, p->small, a, st)
                                     : sw::idisp_launch_mfma<8, false>(p->tscrunch, p->small, a, st);
                if(rc) return rc;
            }
        }
        return SW_OK;
    }
    const bool pf = p->rows_cap <= sw::kPfRows && (nwords & 3) == 0;
    for(int tb0 = 0; tb0 < ntb; tb0 += 65535) {
        const dim3 grid((unsigned)p->tiles.size(), (unsigned)nchunks, (unsigned)std::min(65535, ntb - tb0));
#define SW_ID_LAUNCH(TT, WIDE, PF)                                                                         \
    hipLaunchKernelGGL((sw::idisp_kernel<2, TT, WIDE, PF>), grid, dim3(256), lds, st,                     \
                       static_cast<const uint32_t*>(d_tfb), static_cast<uint32_t*>(d_tdb), p->d_delays,   \
                       p->d_span, p->d_tiles, p->nchans, nwords, p->ndms, p->tscrunch, p->max_delay,      \
                       (long)nsamples, nout, tb0, p->scale, stride_t, stride_f)
        if(p->wide) {
            if(p->tt == 8)
                SW_ID_LAUNCH(8, true, false);
            else
                SW_ID_LAUNCH(4, true, false);
        } else if(p->tt == 16) {
            if(pf)
                SW_ID_LAUNCH(16, false, true);
            else
                SW_ID_LAUNCH(16, false, false);
        } else {
            SW_ID_LAUNCH(4, false, false);
        }
#undef SW_ID_LAUNCH
        SW_LAUNCH_CHECK();
    }
    return SW_OK;
}
