// qw6_prefill.hip -- the MoE FFN for a batch of tokens (prefill, batched
// verification) as grouped fp16-MFMA contractions on gfx950.
//
// qw6 runs its MoE block token by token (qw6_forward_token -> qw6_apply_layer_
// moe, qw6.c:2226-2290; qw6_prefill, qw6.c:2867-2882). With T tokens of top-8
// routing, expert e sees M_e of them; its gate/up/down are then T x K by K x N
// products over the M_e gathered rows. Kernels, in stream order:
//   k_pre_x       one workgroup per token: the optional RMSNorm, the fp16
//                 operands of the input, the shared expert's gate.
//   k_pre_router, k_pre_router_mfma  router logits, when none are given.
//   k_pre_route   one wave per token: softmax top-k (wave_route); without a norm
//                 or with given logits k_pre_x does this, after the router.
//   k_pre_sort    one workgroup: counting sort of the (token, k) pairs by
//                 expert into "entries" and a list of tiles of up to
//                 prefill_tile_entries entries of one expert (the shared
//                 expert last, with every token).
//   k_pre_gemm<0> gate and up for 64 intermediate rows of one tile:
//                 mid[entry] = silu(x.gate) * (x.up).
//   k_pre_gemm<1> down for 128 hidden rows of one tile, times the entry's gate
//                 weight -> ybuf[entry].
//   k_pre_combine out[t] = sum_k ybuf[entry(t, k)] + ybuf[shared entry(t)]
//                 (+ residual), a fixed order: deterministic, no atomics.
//
// Numerics of the contraction (2.1e-7 to 3.7e-7 against 64-bit results, 17 to 2048
// tokens, every format):
//  - weights enter the MFMA exactly, with their sub-block scale folded in where
//    that is exact in fp16 (qw6_f16tile.h);
//  - activations enter as two fp16 parts (22 significant bits; calls of fewer than
//    kPrefill3PartBelow tokens: three, 24 bits), one MFMA each into a sum of its own, scaled by
//    a power of two per token (the input) or per 64 columns of an entry (mid);
//  - products accumulate in fp32, per block (down: per 64 columns), times the block's
//    factor d; the K-quant minimum dmin * m is one more MFMA against the
//    three-part sub-block sums of the represented activations.

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <iterator>
#include <type_traits>

#include "qw6_dev.h"
#include "qw6_f16tile.h"
#include "qw6_moe.h"
#include "qw6_tile.h"

namespace qw6 {
namespace {

__device__ const IqTables g_tabs_pre = make_tables();

constexpr uint32_t kPM = prefill_tile_entries(false);   // entries per tile at most
constexpr uint32_t kPWG = 256;    // threads per workgroup (4 waves)

// ---- input operands ------------------------------------------------------------------

// Sum and maximum of a pair over the workgroup's four waves (every thread gets both).
__device__ __forceinline__ void block_sum_max(float& s, float& m, float (&red)[2][4]) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    s = group_sum<64>(s);
#pragma unroll
    for (uint32_t i = 1; i < 64; i <<= 1) m = fmaxf(m, partner(m, i, lane));
    if (lane == 0) { red[0][wave] = s; red[1][wave] = m; }
    __syncthreads();
    s = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
    m = fmaxf(fmaxf(red[1][0], red[1][1]), fmaxf(red[1][2], red[1][3]));
    __syncthreads();   // red may be written again
}

// Softmax top-k of token t by one wave (lane l of it).
__device__ __forceinline__ void route_token(const PrefillLayer& L, const PrefillWs& ws, const float* logits,
                                            uint32_t t, uint2* scr, uint32_t lane) {
    wave_route(logits + (size_t)t * L.n_experts, L.n_experts, L.top_k, scr,
               ws.pidx + (size_t)t * L.top_k, ws.pw + (size_t)t * L.top_k);
    __builtin_amdgcn_wave_barrier();
    if (lane < L.top_k) {
        const size_t i = (size_t)t * L.top_k + lane;
        if (L.idx_out) L.idx_out[i] = ws.pidx[i];
        if (L.w_out) L.w_out[i] = ws.pw[i];
    }
}
__global__ __launch_bounds__(64) void k_pre_route(PrefillLayer L, PrefillWs ws, const float* __restrict__ logits) {
    __shared__ uint2 scr[kRouteScr];
    route_token(L, ws, logits, blockIdx.x, scr, threadIdx.x);
}

// One workgroup per token: y = rmsnorm(x) * w when the layer has a norm
// (qw6.c:2503-2513; written to xn where the router reads it), y's fp16 parts at
// scale 2^e, their 32-column sums, and the shared entry with its weight
// sigmoid(shared_router . y) (qw6.c:2267-2285). Thread c holds columns
// 8 c .. 8 c + 7 (hidden <= 2048), so the row is read once.
// ROUTE: wave 0 routes the token, too: a launch less (1 us of a 26 us call) where
// the logits don't wait for the norm formed here.
template <bool ROUTE>
__global__ __launch_bounds__(kPWG) void k_pre_x(PrefillLayer L, PrefillWs ws, const float* __restrict__ logits) {
    __shared__ uint2 scr[ROUTE ? kRouteScr : 1];
    __shared__ float red[2][4];
    const uint32_t t = blockIdx.x, c = threadIdx.x, lane = c & 63u;
    const bool on = c < L.hidden / 8;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto load8 = [&](const float* p, float (&o)[8]) {
        const float4 a = ((const float4*)p)[2 * c], b = ((const float4*)p)[2 * c + 1];
        o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
    };
    float w[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, sr[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (on) {
        load8(L.x + (size_t)t * L.hidden, v);
        if (L.norm_w) load8(L.norm_w, w);
        if (L.shared_router) load8(L.shared_router, sr);
    }
    if (L.norm_w) {
        float ss = 0.f, none = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) ss = fmaf(v[i], v[i], ss);
        block_sum_max(ss, none, red);
        const float sc = 1.0f / sqrtf(ss / (float)L.hidden + L.norm_eps);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = v[i] * sc * w[i];
        if (on && !L.logits) {
            float4* o = (float4*)(ws.xn + (size_t)t * L.hidden) + 2 * c;
            o[0] = make_float4(v[0], v[1], v[2], v[3]);
            o[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
    float dot = 0.f, mx = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        dot = fmaf(sr[i], v[i], dot);
        mx = fmaxf(mx, fabsf(v[i]));
    }
    block_sum_max(dot, mx, red);
    float inv;
    const float sc = group_scale(mx, inv);
    float sum;
    auto put = [&](auto pc) {
        constexpr int P = decltype(pc)::value;
        uint4 part[P];
        sum = split8h<P>(v, sc, part);
        uint4* o = (uint4*)(ws.xp + (size_t)t * P * L.hidden) + 32 * P * (c >> 5) + (c & 31u);
#pragma unroll
        for (int p = 0; p < P; p++)
            if (on) o[32 * p] = part[p];
    };
    if (L.three) put(std::integral_constant<int, 3>{});
    else put(std::integral_constant<int, 2>{});
    sum += partner(sum, 1, lane);
    sum += partner(sum, 2, lane);
    if (on && (c & 3u) == 0) ws.xs[(size_t)t * (L.hidden / 32) + (c >> 2)] = split_sum(sum);
    if (c == 0) {
        ws.xinv[t] = inv;
        const uint32_t e = L.T * L.top_k + t;
        ws.ent_tok[e] = t;
        ws.ent_w[e] = L.shared_router ? 1.0f / (1.0f + expf(-dot)) : 1.0f;
    }
    if (ROUTE && c < 64) route_token(L, ws, logits, t, scr, lane);
}

// ---- routing -----------------------------------------------------------------------

// Counting sort of the T * top_k (token, k) pairs by expert, one workgroup.
// Entries of one expert are contiguous; their order inside the expert does
// not affect any result (every entry's output depends on its own row only,
// and the combine sums in (token, k) order). Then the list of tiles of up to pm
// entries of one expert, the shared expert (with every token) last: first the full
// tiles and those of more than 16 entries, then the others, each in the order of the
// experts.
__global__ __launch_bounds__(1024) void k_pre_sort(PrefillLayer L, PrefillWs ws) {
    __shared__ uint32_t cnt[257], off[257], cur[257];
    __shared__ uint32_t pos[2][257];   // an expert's first large tile, its small one
    __shared__ uint32_t n_big;
    const uint32_t tid = threadIdx.x, nthr = blockDim.x;
    const uint32_t ne = L.T * L.top_k, E = L.n_experts;
    const uint32_t pm = prefill_tile_entries(L.three);   // a power of two
    // Every global load a thread needs goes out before its first wait: its
    // PT (token, k) pairs' experts and gate weights. Calls beyond PT pairs per
    // thread (2048 tokens of top-8) reload per chunk.
    constexpr uint32_t PT = 16;
    const uint32_t chunk = PT * nthr;
    uint32_t ev[PT];
    float wv[PT];
#pragma unroll
    for (uint32_t u = 0; u < PT; u++) {
        if (u * nthr >= ne) break;
        const uint32_t i = u * nthr + tid;
        ev[u] = i < ne ? ws.pidx[i] : 0u;
        wv[u] = i < ne ? ws.pw[i] : 0.f;
    }
    if (tid <= E) cnt[tid] = tid == E && L.sg.p ? L.T : 0u;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < ne; c0 += chunk) {
        if (c0) {
#pragma unroll
            for (uint32_t u = 0; u < PT; u++) {
                if (c0 + u * nthr >= ne) break;
                const uint32_t i = c0 + u * nthr + tid;
                ev[u] = i < ne ? ws.pidx[i] : 0u;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < PT; u++) {
            if (c0 + u * nthr >= ne) break;
            if (c0 + u * nthr + tid < ne) atomicAdd(&cnt[ev[u]], 1u);
        }
    }
    __syncthreads();
    const uint32_t wave = tid >> 6, lane = tid & 63u;
    if (wave == 0) {   // exclusive scan of the counts
        uint32_t run = 0;
        for (uint32_t e0 = 0; e0 < E; e0 += 64) {
            const uint32_t e = e0 + lane;
            const uint32_t c = e < E ? cnt[e] : 0u;
            const uint32_t sc = wave_scan_incl(c, lane);
            if (e < E) off[e] = cur[e] = run + sc - c;
            run += __builtin_amdgcn_readlane(sc, 63);
        }
        if (lane == 0) off[E] = run;
    } else if (wave < 3) {   // and of the tiles: wave 1 the large ones, wave 2 the others
        uint32_t run = 0;
        for (uint32_t e0 = 0; e0 <= E; e0 += 64) {
            const uint32_t e = e0 + lane, c = e <= E ? cnt[e] : 0u, rem = c & (pm - 1);
            const uint32_t nt = wave == 1 ? (c - rem) / pm + (rem > 16 ? 1u : 0u) : rem != 0 && rem <= 16 ? 1u : 0u;
            const uint32_t sc = wave_scan_incl(nt, lane);
            if (e <= E) pos[wave - 1][e] = run + sc - nt;
            run += __builtin_amdgcn_readlane(sc, 63);
        }
        if (lane == 0) ws.n_tiles[wave - 1] = run;
        if (lane == 0 && wave == 1) n_big = run;
    }
    __syncthreads();
    for (uint32_t c0 = 0; c0 < ne; c0 += chunk) {
        if (ne > chunk) {   // the registers hold the last chunk: reload
#pragma unroll
            for (uint32_t u = 0; u < PT; u++) {
                if (c0 + u * nthr >= ne) break;
                const uint32_t i = c0 + u * nthr + tid;
                ev[u] = i < ne ? ws.pidx[i] : 0u;
                wv[u] = i < ne ? ws.pw[i] : 0.f;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < PT; u++) {
            if (c0 + u * nthr >= ne) break;
            const uint32_t i = c0 + u * nthr + tid;
            if (i >= ne) continue;
            const uint32_t p = atomicAdd(&cur[ev[u]], 1u);
            if (p >= ne) continue;   // cannot happen: the counts bound every expert's range
            ws.ent_tok[p] = i / L.top_k;
            ws.ent_w[p] = wv[u];
            ws.ent_pos[i] = p;
        }
    }
    // four threads per expert, all for the shared one
    const uint32_t cap = prefill_tiles_max(L.T, L.top_k, E, L.three);
    auto put = [&](uint32_t e, uint32_t first, uint32_t step) {
        const uint32_t c = cnt[e];
        for (uint32_t j = first; j * pm < c; j += step) {
            const uint32_t m = min(pm, c - j * pm), o = m == pm || m > 16 ? pos[0][e] + j : n_big + pos[1][e];
            if (o < cap) ws.tiles[o] = make_uint4(e, off[e] + j * pm, m, 0u);
        }
    };
    if (tid / 4 < E) put(tid / 4, tid % 4, 4);
    put(E, tid, nthr);
}

// ---- the grouped contraction --------------------------------------------------------

constexpr uint32_t kGW = 8;              // waves per workgroup of k_pre_gemm, 16 weight rows each
constexpr uint32_t kMidRows = 8 * kGW;   // intermediate rows of an item (MODE 0): one scale group of mid
constexpr uint32_t kOutRows = 16 * kGW;  // hidden rows of an item (MODE 1)

// Shared memory of k_pre_gemm: the stages of the tile's A rows (gemm_item), 512 bytes
// a row, piece i of row m at slot i ^ (m % 16), so that eight rows' reads of one piece
// take all banks; the waves' raw weight blocks; by format, two stages of the sub-block sums
// (K-quants with minimums) or the IQ lattice; the entries' factors (the input's
// reciprocal scale; MODE 1: the mid scales per 64 columns, the gate weight where there is
// room). MODE 0's results take the place of the A rows.
constexpr uint32_t kStageRow = 512;
constexpr uint32_t kGroupA = 16u * kStageRow;   // a row group of A
constexpr uint32_t kStageA = kPM * kStageRow;
constexpr uint32_t kStageS = kPM * 64u;
constexpr uint32_t kMidLd = kMidRows + 4;
constexpr uint32_t kOffW = 3u * kStageA;
static_assert(kPM * kMidLd * 4u <= kOffW, "MODE 0's results fit");
__host__ __device__ constexpr uint32_t off_tab(int f) { return kOffW + kGW * 16u * 16u * stage_stride(f); }
__host__ __device__ constexpr uint32_t off_fac(int f) {
    return off_tab(f) + (f == F_Q4K || f == F_Q5K ? 2u * kStageS : f16_grid_bytes(f));
}
template <int MODE>
__host__ __device__ constexpr uint32_t gemm_lds(int f, uint32_t inter) {
    return off_fac(f) + 4u * kPM * (MODE == 1 ? inter / 64u : 1u);
}
constexpr uint32_t kLdsHalf = 80u * 1024u;
static_assert(gemm_lds<0>(F_Q4K, 2048) <= kLdsHalf && gemm_lds<0>(F_Q5K, 2048) <= kLdsHalf &&
              gemm_lds<0>(F_Q6K, 2048) <= kLdsHalf && gemm_lds<0>(F_IQ2XXS, 2048) <= kLdsHalf &&
              gemm_lds<0>(F_IQ2S, 2048) <= kLdsHalf && gemm_lds<0>(F_IQ3S, 2048) <= kLdsHalf &&
              gemm_lds<1>(F_Q4K, 2048) <= kLdsHalf && gemm_lds<1>(F_Q5K, 2048) <= kLdsHalf &&
              gemm_lds<1>(F_Q6K, 2048) <= kLdsHalf && gemm_lds<1>(F_IQ3S, 2048) <= kLdsHalf &&
              gemm_lds<1>(F_IQ2S, 2048) <= kLdsHalf && gemm_lds<1>(F_IQ2XXS, 2048) <= kLdsHalf,
              "two workgroups per CU at every size");

// At most N of this wave's vector memory operations still in flight.
template <uint32_t N>
__device__ __forceinline__ void wait_loads() {
    __builtin_amdgcn_s_waitcnt((N & 15u) | ((N >> 4) << 14) | 0x0f70u);   // vmcnt; expcnt, lgkmcnt not waited
}
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07fu); }   // lgkmcnt(0) only
// Workgroup barrier without a memory fence (which would wait for every load
// in flight); what the other waves read after it is waited for by hand before it.
__device__ __forceinline__ void bare_barrier() { asm volatile("s_barrier" ::: "memory"); }

template <int MODE>
__host__ __device__ inline uint32_t gemm_row_blocks(uint32_t hidden, uint32_t inter) {
    return MODE == 0 ? inter / kMidRows : hidden / kOutRows;
}

// A uniform load of data that the kernel does not write, emitted as a scalar load.
template <typename T>
__device__ __forceinline__ T ld_uniform(const T* p) {
    return *(const __attribute__((address_space(4))) T*)(uintptr_t)p;
}

// One item: a tile's entries (at most 16 MT / R) against one row block of their expert's
// matrix (format F), 16 rows per wave, activations in P parts.
//
// Two workgroups of eight waves share a CU, so 256 rows are all that it has in
// flight: a block's 144 bytes (Q4_K) start inside a 128-byte line for 7 of 8 blocks,
// so most lines are read for two blocks, and the second read finds the line in
// the XCD's 4 MB L2 only if its 32 CUs bring in less than that between (with 512
// rows a CU, 1.9 times the weights' bytes were fetched). All loads are coalesced
// (adjacent lanes read adjacent 16 B): loads whose lanes each read a row of
// their own, as the MFMA operands want them, take the vector cache four times the
// accesses. The weights come through registers and the wave's own rows of LDS (no
// barrier), requested a block ahead; the A rows by direct-to-LDS loads, a block ahead
// (32-entry tiles: two half blocks), one barrier per stage.
//
// Bound (rocprofv3 counters, gate/up; busy shares of vector units, LDS, matrix units, HBM
// at 5.1 TB/s): 33 tokens Q4_K by HBM (41, 25, 10, 74%); 100 tokens IQ2_XXS by the
// lattice reads (50, 51, 8, 32%; 44% of the LDS cycles are bank conflicts); 512 tokens Q4_K
// nothing alone (50, 35, 19, 62%; the barriers keep them from overlapping); 2048
// tokens by decoding and the LDS reads of A (60, 46, 29, 38%; each wave reads the whole
// tile for its 16 rows). Measured, us, 256 experts top-8 with the shared expert, hidden
// 2048, inter 512, gate/up + down (bf16 parts -> two fp16 parts in one unit -> now, with
// parts 2^11 apart, three of them at 33 tokens):
//   33 tokens Q4_K / Q6_K      55.3 + 40.9 -> 52.3 + 38.3 -> 39.1 + 31.4
//   100 tokens Q4_K / Q6_K                    70.0 + 52.8 -> 61.0 + 49.1
//   100 tokens IQ2_XXS / IQ3_S                82.8 + 50.7 -> 75.4 + 46.0
//   512 tokens Q4_K / Q6_K     132.5 + 100.5 -> 121 + 88 -> 113 + 88.7
//   509 tokens IQ2_XXS, IQ3_S, IQ2_S  144 + 120 -> 145 + 94 -> 134 + 86
//   2048 tokens Q4_K / Q6_K    342 + 277 -> 321 + 239 -> 309 + 246
// Gained by: the parts as rows of small tiles (R > 1), loads that the compiler does not
// wait for (below), whole-block stages. Slower than with the parts in one unit: Q6_K gate/up
// from 512 tokens, 2 to 4% (its scales multiply every step's sums, now one per part).
// Tried and slower: 32x32x16 MFMA with 32 rows a wave, 64 entries a tile and one
// persistent workgroup per CU (79 + 64, 151 + 133, 309 + 252); each step's operands read
// a step ahead (Q6_K spills: down 144 at 512 tokens); unaligned LDS reads of the
// codes (down 136); leaving out the loads of rows past the tile by a branch (the
// compiler then waits for every load in flight).
//
// MODE 0: gate and up, 8 rows of each: lanes n < 8
// hold gate row n, lanes n >= 8 up row 15 - n (partner pairs mirror lanes). MODE 1: down.
template <int MODE, int F, int MT, int P, int R>
__device__ __forceinline__ void gemm_item(const PrefillLayer& L, const PrefillWs& ws, const uint8_t* m0,
                                          const uint8_t* m1, uint32_t ent0, uint32_t cnt, uint32_t yb,
                                          uint8_t* smem) {
    constexpr uint32_t bb = fmt_block_bytes(F);
    constexpr uint32_t NCH = raw_chunks(F), RS = stage_stride(F);
    constexpr bool kWhole = R > 1 || MT == 1;   // a stage is a block, else half a block
    static_assert(R == 1 || R == (P == 3 ? 4 : 2), "parts in rows");
    static_assert(kWhole || P == 2, "a row holds half a block of two parts");
    // a wave's loads of a block's weights; of a stage of A rows (one per row group)
    constexpr uint32_t NW = (16 * NCH + 63) / 64, NA = kWhole && R == 1 ? P : MT;
    constexpr uint32_t kStg = kWhole ? NA * kGroupA : kStageA;   // bytes from stage to stage
    static_assert((kWhole ? 2 : 3) * kStg <= kOffW, "the stages fit");
    constexpr int VL = 4 / R;   // entries of a lane's four sums (one row group)
    constexpr uint32_t kFacLd = kWhole ? 16 : kPM;   // entries of a row of scales
    constexpr bool kAl = F == F_Q4K || F == F_Q5K;   // blocks are 16-byte aligned
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t n = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t K = MODE == 0 ? L.hidden : L.inter, nblk = K / 256, rb = nblk * bb;
    uint8_t* const tab = smem + off_tab(F);
    float* const fac = (float*)(smem + off_fac(F));
    float* const scl = fac + (kWhole ? kFacLd : 0);   // MODE 1: [64-column group][entry] scales, a whole-block item's after its weights
    const uint32_t wraw = kOffW + wave * (256u * RS);

    // the wave's rows: MODE 0: 0 .. 7 at b0 + row * rb, 8 .. 15 at b1 + row * rb (uniform)
    const uint32_t r0 = MODE == 0 ? kMidRows * yb + 8 * wave : kOutRows * yb + 16 * wave;
    const uint8_t* const b0 = m0 + (size_t)r0 * rb;
    const uint8_t* const b1 = MODE == 0 ? m1 + (size_t)r0 * rb - (size_t)8 * rb : b0;
    // Load i takes piece c % NCH of row c / NCH, c = 64 i + lane (c < 256, so the
    // division by multiplication is exact); lanes past the last repeat it.
    u32x4 fl[NW];
    auto load_w = [&](uint32_t kb) {
#pragma unroll
        for (uint32_t i = 0; i < NW; i++) {
            const uint32_t c = min(64 * i + lane, 16 * NCH - 1), row = (c * (65536u / NCH + 1u)) >> 16;
            uint32_t o = row * (rb - 16 * NCH) + 16 * c + kb * bb;   // row * rb + 16 * piece + kb * bb
            if (!kAl) {
                // 16-byte pieces from the one that the block starts in (the matrix is
                // 16-byte aligned); never past the one that it ends in
                const uint32_t last = (row * rb + kb * bb + bb - 1) & ~15u;
                o &= ~15u;
                if (F == F_IQ3S) o = min(o, last);   // 7 or 8 pieces; the other formats' blocks take NCH
            }
            const uint8_t* const src = MODE == 1 ? b0 : row < 8 ? b0 : b1;
            fl[i] = ld_global<u32x4>(src + (uint64_t)o);
        }
    };
    auto store_w = [&]() {
#pragma unroll
        for (uint32_t i = 0; i < NW; i++) {
            const uint32_t c = min(64 * i + lane, 16 * NCH - 1), row = (c * (65536u / NCH + 1u)) >> 16;
            *(u32x4*)(smem + wraw + 16 * (RS == NCH ? c : c + row)) = fl[i];
        }
    };

    // A rows: load i of wave w takes rows 2 w, 2 w + 1 of row group i. A stage is
    // - half a block, a row an entry's two parts, a group 16 entries (MT = 2, R = 1);
    // - a block, a row an entry's part i, a group one part (MT = 1, R = 1);
    // - a block, row m part m % R of entry m / R (R > 1): tiles of up to 16 MT / R entries
    //   take MT MFMAs a step and as many reads of A, not P.
    // All waves issue the same number of loads, so that the waits below hold for each; rows
    // past the tile are 16 bytes of its last one (a row of A makes a row of D, so what they
    // hold changes no result), one line for the cache to look up.
    uint32_t ar[NA], as = 0;
    auto a_entry = [&](uint32_t i) {   // the lane's entry in load i
        const uint32_t r = 2 * wave + lane / 32;
        return kWhole && R == 1 ? r : (16 * i + r) / R;
    };
    const uint8_t* const abase = (const uint8_t*)(MODE == 0 ? ws.xp : ws.mp + (size_t)ent0 * P * K);
    const uint8_t* const sbase = (const uint8_t*)(MODE == 0 ? ws.xs : ws.ms + (size_t)ent0 * (K / 32));
    auto stage_a = [&](uint32_t kb, uint32_t h, uint32_t buf) {   // (whole blocks: h = 0)
#pragma unroll
        for (uint32_t i = 0; i < NA; i++)
            __builtin_amdgcn_global_load_lds((glb_void_t*)(abase + kb * (512 * P) + 256 * h + (uint64_t)ar[i]),
                                             (lds_void_t*)(smem + buf * kStg + (kGW * i + wave) * 1024), 16, 0, 0);
        if constexpr (has_min<F>()) {
            if (h == 0 && wave < MT)
                __builtin_amdgcn_global_load_lds((glb_void_t*)(sbase + kb * 64 + (uint64_t)as),
                                                 (lds_void_t*)(tab + (kb & 1u) * kStageS + wave * 1024), 16, 0, 0);
        }
    };

    // The start. Loads land in the order of their issue, so the short ones that others or
    // the first steps wait for (the tile's tokens, the lattice, the scales) go out
    // before the weights, and what only the end needs is kept in a register till then.
    F16Grid<is_iq(F) ? F : (int)F_IQ3S, 64 * kGW> grid;
    if constexpr (is_iq(F)) grid.load(g_tabs_pre);
    uint32_t tok[NA], tok_s = 0, tok_f = 0;
#pragma unroll
    for (uint32_t i = 0; i < NA; i++) {
        const uint32_t e = min(a_entry(i), cnt - 1);
        tok[i] = MODE == 0 ? ws.ent_tok[ent0 + e] : e;
    }
    if constexpr (has_min<F>()) {   // waves 0 .. MT - 1 load the sums of rows 16 w ..
        const uint32_t e = min((16 * min(wave, MT - 1u) + lane / 4) / R, cnt - 1);
        tok_s = MODE == 0 ? ws.ent_tok[ent0 + e] : e;
    }
    const uint32_t own = ent0 + min(tid, cnt - 1), ng = L.inter / 64;
    float f_own = 0.f, sc[2] = {0.f, 0.f};
    if (MODE == 0) tok_f = ws.ent_tok[own];
    else if (kWhole) f_own = ws.ent_w[own];
    constexpr uint32_t NS = kFacLd / 16;   // at most 32 groups for 512 threads
    if (MODE == 1) {
#pragma unroll
        for (uint32_t u = 0; u < NS; u++) {
            const uint32_t i = u * 64 * kGW + tid, m = i % kFacLd, gr = i / kFacLd;
            if (gr < ng) sc[u] = ws.minv[(size_t)(ent0 + min(m, cnt - 1)) * ng + gr];
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_w(0);
    __builtin_amdgcn_sched_barrier(0);
    if (MODE == 0) asm volatile("" : "+v"(tok_s), "+v"(tok_f));   // waited for here, with the weights behind them in flight
#pragma unroll
    for (uint32_t i = 0; i < NA; i++) {
        const uint32_t r = 2 * wave + lane / 32, j = (lane & 31u) ^ r;   // the row in its group, its piece
        const uint32_t part = R > 1 ? (16 * i + r) % R : i;
        const uint32_t o = kWhole ? part * 512 + 16 * j : (j / 16) * 512 + 16 * (j % 16);
        ar[i] = tok[i] * (2 * P * K) + (a_entry(i) < cnt && (!kWhole || part < P) ? o : 0u);
    }
    as = tok_s * (K / 4) + 16 * (lane & 3u);
    stage_a(0, 0, 0);
    if (!kWhole) stage_a(0, 1, 1);
    if (MODE == 0) f_own = ws.xinv[tok_f];
    if constexpr (is_iq(F)) grid.store(tab);
    if (MODE == 1) {
        if (kWhole && tid < kFacLd) fac[tid] = f_own;
#pragma unroll
        for (uint32_t u = 0; u < NS; u++) {
            const uint32_t i = u * 64 * kGW + tid, m = i % kFacLd, gr = i / kFacLd;
            if (gr < ng) scl[gr * kFacLd + m] = sc[u];
        }
    }

    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    constexpr int PS = folds<F>() && R == 1 ? P : 1;
    // results so far (VL of four); products of the block (MODE 0) or of 64 columns in its unit
    f32x4 acc[MT], blk[PS][MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        acc[mt] = zero;
#pragma unroll
        for (int p = 0; p < PS; p++) blk[p][mt] = zero;
    }
    Head<F> hd;
    const uint32_t row = MODE == 0 && n >= 8 ? 23 - n : n;   // the lane's row among the staged ones
    uint32_t buf = 0;
    auto joined = [](const auto& c, int mt, int j) {   // the parts' sums of the lane's entry j
        constexpr size_t N = R > 1 ? P : std::extent_v<std::remove_reference_t<decltype(c)>>;
        float v[N];
#pragma unroll
        for (size_t p = 0; p < N; p++) v[p] = R > 1 ? c[0][mt][R * j + p] : c[R > 1 ? 0 : p][mt][j];
        return join(v);
    };
    // Step s of block kb, staged at w; its A rows are in stage buf.
    auto step = [&](uint32_t kb, const LdsBlock& w, int s) {
        const uint8_t* const A = smem + buf * kStg + kStageRow * n;
        constexpr int NP = R > 1 ? 1 : P;   // operands per row group
        u32x4 a[MT][NP];
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int p = 0; p < NP; p++)
                a[mt][p] = *(const u32x4*)(kWhole ? A + kGroupA * (R > 1 ? mt : p) + 16 * ((4 * s + g) ^ n)
                                                  : A + kGroupA * mt + 16 * ((16 * p + 4 * (s & 3) + g) ^ n));
        const Codes<F> q = read_codes<F>(w, s, g);
        const u32x4 b = b_operand<F>(hd, q, look_up<F>(q, hd, s, g, tab), w, s, g);
        if constexpr (folds<F>()) {
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) blk[p][mt] = mfma_h(a[mt][p], b, blk[p][mt]);
        } else {
            const float ds = run_scale(hd, s) * h2f(hd.d);
            f32x4 c[NP][MT];
#pragma unroll
            for (int p = 0; p < NP; p++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) c[p][mt] = mfma_h(a[mt][p], b, zero);
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int j = 0; j < VL; j++) blk[0][mt][j] = fmaf(ds, joined(c, mt, j), blk[0][mt][j]);
        }
        const bool sums = MODE == 1 ? (s & 1) : s == 7;   // the sums of these columns are complete
        if (sums) {
            const float d = folds<F>() ? block_scale<F>(hd) : 1.f;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                f32x4 v;
#pragma unroll
                for (int j = 0; j < VL; j++) v[j] = folds<F>() ? joined(blk, mt, j) * d : blk[0][mt][j];
                if constexpr (has_min<F>()) {
                    const float dm = -block_min<F>(hd);
                    u32x4 m = min_operand<F>(hd, g);
                    if (MODE == 1 && g != (uint32_t)(s >> 1)) m = u32x4{0, 0, 0, 0};
                    const f32x4 mn = mfma_h(*(const u32x4*)(tab + (kb & 1u) * kStageS + 1024 * mt + 64 * n + 16 * g), m, zero);
#pragma unroll
                    for (int j = 0; j < VL; j++) v[j] = fmaf(dm, mn[R * j], v[j]);
                }
                f32x4 sj = {1.f, 1.f, 1.f, 1.f};
                if (MODE == 1) {
                    const float* const f = scl + (4 * kb + (s >> 1)) * kFacLd + (16 * mt + 4 * g) / R;
                    if (R == 1) sj = *(const f32x4*)f;
                    else
#pragma unroll
                        for (int j = 0; j < VL; j++) sj[j] = f[j];
                }
#pragma unroll
                for (int j = 0; j < VL; j++) acc[mt][j] = MODE == 1 ? fmaf(sj[j], v[j], acc[mt][j]) : acc[mt][j] + v[j];
#pragma unroll
                for (int p = 0; p < PS; p++) blk[p][mt] = zero;
            }
        }
    };
    // The blocks but the last, then the last, which requests no loads. With that as a condition
    // in one loop the compiler could not tell how many loads follow the weights', and
    // waited for all of them before it stored the weights, the A rows requested a moment
    // before among them (a lambda in place of the outer loop spills).
#pragma unroll
    for (int last = 0; last < 2; last++) {
        for (uint32_t kb = last ? nblk - 1 : 0; kb < (last ? nblk : nblk - 1); kb++) {
            const bool more = !last;
            if (kWhole) {   // requested with the block's weights
                wait_lds();
                wait_loads<0>();
                bare_barrier();
                store_w();
                if (more) {
                    stage_a(kb + 1, 0, buf ^ 1u);
                    load_w(kb + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                const LdsBlock w(smem, wraw + 16 * RS * row + (kAl ? 0u : (row * rb + kb * bb) & 15u));
                read_head<F>(hd, w, g);
#pragma unroll
                for (int s = 0; s < 8; s++) step(kb, w, s);
                __builtin_amdgcn_sched_barrier(0);
                buf ^= 1u;
                continue;
            }
            wait_lds();
            wait_loads<NA>();   // first half's A rows and the weights; the second half's A rows may be in flight
            bare_barrier();     // ... of every wave; and the stage before the running one is free
            const uint32_t b2 = buf == 0 ? 2 : buf - 1;
            if (MODE == 1 && last) f_own = ws.ent_w[own];
            store_w();
            if (more) {
                stage_a(kb + 1, 0, b2);
                load_w(kb + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
            const LdsBlock w(smem, wraw + 16 * RS * row + (kAl ? 0u : (row * rb + kb * bb) & 15u));   // (8 rows are a multiple of 16 bytes)
            read_head<F>(hd, w, g);
#pragma unroll
            for (int s = 0; s < 4; s++) step(kb, w, s);
            __builtin_amdgcn_sched_barrier(0);
            wait_lds();
            if (more) wait_loads<NA + NW>();   // the next block's first A rows and weights, at least
            else wait_loads<0>();
            if (MODE == 1 && last) {   // the gate weights, in the stage that the last block leaves free
                if (tid < kPM) ((float*)(smem + b2 * kStageA))[tid] = f_own;
                wait_lds();
            }
            bare_barrier();
            if (more) stage_a(kb + 1, 1, buf);
            buf = buf == 2 ? 0 : buf + 1;
#pragma unroll
            for (int s = 4; s < 8; s++) step(kb, w, s);
            __builtin_amdgcn_sched_barrier(0);
            buf = buf == 2 ? 0 : buf + 1;
        }
    }

    // Results: lane holds entries (16 mt + 4 g) / R + j of row n.
    if constexpr (MODE == 0) {
        // mid = silu(gate) * up. Gate rows are in lanes n < 8, their up rows in 15 - n: the former
        // form two of four entries' results, the latter the other two. Then, sixteen
        // threads an entry, the fp16 parts of its 64 columns at one scale and their
        // 32-column sums.
        float* const mid = (float*)smem;   // [entry][kMidLd]
        const bool up = n >= 8;
        if (tid < 16 * MT) fac[tid] = f_own;
        wait_lds();
        bare_barrier();   // every wave has read its A rows
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const uint32_t e0 = (16 * mt + 4 * g) / R;
            float v[VL];
#pragma unroll
            for (int j = 0; j < VL; j++) v[j] = acc[mt][j] * fac[e0 + j];
            constexpr int VH = (VL + 1) / 2;   // (a single one: the gate lanes form it)
#pragma unroll
            for (int j = 0; j < VH; j++) {
                const float got = partner(up ? v[j] : v[VL / 2 + j], 8, lane);
                const float gv = up ? got : v[j], uv = up ? v[VL / 2 + j] : got;
                if (VL > 1 || !up)
                    mid[(e0 + (up ? VL / 2 : 0) + j) * kMidLd + 8 * wave + (up ? 15 - n : n)] = gv / (1.0f + expf(-gv)) * uv;
            }
        }
        wait_lds();
        bare_barrier();
        const uint32_t m = tid / 16, c4 = tid % 16;
        if (m < 16 * MT / R) {   // (whole waves)
            const float4 v = *(const float4*)(mid + m * kMidLd + 4 * c4);
            float mx = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
#pragma unroll
            for (uint32_t x = 1; x < 16; x <<= 1) mx = fmaxf(mx, partner(mx, x, lane));
            float inv;
            const float s2 = group_scale(mx, inv);
            uint16_t h[4][P];   // stored order: columns 0, 2, 1, 3
            float sum = (split_h<P>(v.x * s2, h[0]) + split_h<P>(v.y * s2, h[2])) +
                        (split_h<P>(v.z * s2, h[1]) + split_h<P>(v.w * s2, h[3]));
#pragma unroll
            for (uint32_t x = 1; x < 8; x <<= 1) sum += partner(sum, x, lane);
            if (m < cnt) {
                const size_t e = ent0 + m;
                const uint32_t col = kMidRows * yb;
                uint2* o = (uint2*)(ws.mp + e * P * L.inter + (col >> 8) * (256 * P) + (col & 255u)) + c4;
#pragma unroll
                for (int p = 0; p < P; p++)
                    o[64 * p] = make_uint2(h[0][p] | ((uint32_t)h[1][p] << 16), h[2][p] | ((uint32_t)h[3][p] << 16));
                if ((c4 & 7u) == 0) ws.ms[e * (L.inter / 32) + 2 * yb + c4 / 8] = split_sum(sum);
                if (c4 == 0) ws.minv[e * (L.inter / 64) + yb] = inv;
            }
        }
    } else {
        const float* const wt = kWhole ? fac : (const float*)(smem + buf * kStageA);   // (buf: b2 of the last block)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int j = 0; j < VL; j++) {
                const uint32_t m = (16 * mt + 4 * g) / R + j;
                if (m < cnt) ws.ybuf[(size_t)(ent0 + m) * L.hidden + r0 + n] = wt[m] * acc[mt][j];
            }
    }
}

// The item's form by its entries: the fewest products and reads of A a step. One row
// group of parts for up to 4 (three parts) or 8 entries, two for up to 8; else a product
// per part, and 32 entries a tile from 17 on (two parts), which share one decoding.
// Against a product per part throughout: 33 tokens Q4_K 59.2 + 43.7 -> 43.7 + 33.5 us,
// 100 tokens IQ2_XXS / IQ3_S 81.1 + 49.7 -> 73.2 + 44.2.
template <int MODE, int F, int P>
__device__ __forceinline__ void gemm_tile(const PrefillLayer& L, const PrefillWs& ws, const uint8_t* m0, const uint8_t* m1,
                                          uint32_t ent0, uint32_t cnt, uint32_t yb, uint8_t* smem) {
    if constexpr (P == 3) {
        if (cnt <= 4) gemm_item<MODE, F, 1, 3, 4>(L, ws, m0, m1, ent0, cnt, yb, smem);
        else if (cnt <= 8) gemm_item<MODE, F, 2, 3, 4>(L, ws, m0, m1, ent0, cnt, yb, smem);
        else gemm_item<MODE, F, 1, 3, 1>(L, ws, m0, m1, ent0, cnt, yb, smem);
    } else {
        if (cnt <= 8) gemm_item<MODE, F, 1, 2, 2>(L, ws, m0, m1, ent0, cnt, yb, smem);
        else if (cnt <= 16) gemm_item<MODE, F, 1, 2, 1>(L, ws, m0, m1, ent0, cnt, yb, smem);
        else gemm_item<MODE, F, 2, 2, 1>(L, ws, m0, m1, ent0, cnt, yb, smem);
    }
}

// One launch per matrix kind over every (tile, row block) item, whatever the
// formats: a workgroup reads its tile's format and branches (uniformly).
// Workgroup p runs on XCD p % 8 (round-robin dispatch). An XCD takes its contiguous
// eighth of the large tiles, then of the small ones: the row blocks of one tile (same A
// rows) and the large tiles of one expert (same weights) share its L2, all XCDs
// have the same work, and the last workgroups are short.
template <int MODE, int P>
__global__ __launch_bounds__(64 * kGW, 4) void k_pre_gemm(PrefillLayer L, PrefillWs ws) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t ny = gemm_row_blocks<MODE>(L.hidden, L.inter), x = blockIdx.x % 8, yb = blockIdx.x / 8 % ny;
    const uint32_t n0 = ld_uniform(ws.n_tiles), n1 = ld_uniform(ws.n_tiles + 1);
    const uint32_t big = x * n0 / 8, nb = (x + 1) * n0 / 8 - big, small = x * n1 / 8, ns = (x + 1) * n1 / 8 - small;
    const uint32_t it = blockIdx.x / 8 / ny;
    if (it >= nb + ns) return;
    const u32x4 tile = ld_uniform((const u32x4*)ws.tiles + (it < nb ? big + it : n0 + small + it - nb));
    const uint32_t e = tile.x;
    const bool shared = e == L.n_experts;
    constexpr int k = MODE == 0 ? 0 : 2;
    const int f = shared ? (MODE == 0 ? L.sg.fmt : L.sd.fmt) : L.pk[k].regular ? L.pk[k].fmt : ld_uniform(&L.experts[e].fmt[k]);
    const uint8_t* const m0 = shared ? (MODE == 0 ? L.sg.p : L.sd.p)
                              : L.pk[k].regular ? L.pk[k].base + L.pk[k].stride * e : ld_uniform(&L.experts[e].p[k]);
    const uint8_t* const m1 = MODE == 1 ? nullptr
                              : shared ? L.su.p
                              : L.pk[1].regular ? L.pk[1].base + L.pk[1].stride * e : ld_uniform(&L.experts[e].p[1]);
#define QW6_ITEM(FMT)                                                                          \
    case FMT:                                                                                  \
        gemm_tile<MODE, FMT, P>(L, ws, m0, m1, tile.y, tile.z, yb, smem);                      \
        break;
    switch (f) {
        QW6_ITEM(F_Q4K)
        QW6_ITEM(F_Q5K)
        QW6_ITEM(F_Q6K)
        QW6_ITEM(F_IQ2XXS)
        QW6_ITEM(F_IQ2S)
        QW6_ITEM(F_IQ3S)
        default: break;
    }
#undef QW6_ITEM
}

// out[t] = sum_k ybuf[entry(t, k)] + ybuf[shared entry(t)] (+ residual); the
// gate weights were applied by the down kernel. Selection order, shared last,
// as qw6.c:2263, 2284.
__global__ __launch_bounds__(256) void k_pre_combine(PrefillLayer L, PrefillWs ws) {
    const uint32_t t = blockIdx.x;
    uint32_t pos[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; k++) pos[k] = k < L.top_k ? ws.ent_pos[(size_t)t * L.top_k + k] : 0u;
    const bool sh = L.sg.p != nullptr;
    const uint32_t se = L.T * L.top_k + t;
    const uint32_t n4 = L.hidden / 4;
    for (uint32_t i = blockIdx.y * 256 + threadIdx.x; i < n4; i += 256 * gridDim.y) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (uint32_t k = 0; k < 8; k++)
            if (k < L.top_k) {
                const float4 y = ((const float4*)(ws.ybuf + (size_t)pos[k] * L.hidden))[i];
                v.x += y.x; v.y += y.y; v.z += y.z; v.w += y.w;
            }
        if (sh) {
            const float4 y = ((const float4*)(ws.ybuf + (size_t)se * L.hidden))[i];
            v.x += y.x; v.y += y.y; v.z += y.z; v.w += y.w;
        }
        if (L.residual) {
            const float4 r = ((const float4*)(L.residual + (size_t)t * L.hidden))[i];
            v.x += r.x; v.y += r.y; v.z += r.z; v.w += r.w;
        }
        ((float4*)(L.out + (size_t)t * L.hidden))[i] = v;
    }
}

// Router logits of TM tokens and TN experts (16 or 32 each) on the fp32 matrix
// cores. Wave w takes the w-th eighth of hidden, in chunks of 32 columns (a 128-byte
// line of each row) loaded straight to LDS, one chunk ahead; the waves need no barrier
// until their sums meet at the end. Lane (m, g) = (l % 16, l / 16) multiplies
// columns 16 h + 4 g + k of a chunk in step (h, k), the same for both operands, so it
// reads them as float4. Piece p of row r is kept at slot p ^ (r % 8): eight rows' reads of
// one piece take all banks.
//
// Every product and sum is fp32: four products per MFMA, each from a zero sum, the
// eight of a chunk added pairwise, the chunks in turn, the waves pairwise. Against 64-bit
// sums (hidden 2048, N(0, 1) inputs) the logits' relative RMS error is 9.7e-8, 1.2e-7
// with k_pre_router; with two running sums per wave it was 2.1e-7.
//
// Bound by the fp32 matrix rate (a lone workgroup takes as long per MFMA as a full
// chip): 256 experts, hidden 2048, us: T = 64: 6.1, 128: 6.3, 512: 10.6, 2048: 32, where
// k_pre_router, which reads the router for every four tokens, takes 8.1, 13.4, 46, 168.
template <int TM, int TN>
__global__ __launch_bounds__(512) void k_pre_router_mfma(const float* __restrict__ router, const float* __restrict__ x,
                                                         float* logits, uint32_t hidden, uint32_t n_experts,
                                                         uint32_t T) {
    constexpr uint32_t ROWS = TM + TN, STAGE = ROWS * 128, NL = ROWS / 8;   // a chunk's bytes and loads per wave
    constexpr int MM = TM / 16, NN = TN / 16;
    __shared__ __attribute__((aligned(16))) uint8_t smem[8 * 2 * STAGE];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, m = lane & 15u, g = lane >> 4;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup p runs on XCD p % 8: token tiles p % 8, p % 8 + 8, ..., each with all
    // experts, so that an L2 reads its tokens once (the router is 2 MB).
    const uint32_t ne = (n_experts + TN - 1) / TN, i8 = blockIdx.x / 8;
    const uint32_t t0 = TM * (blockIdx.x % 8 + 8 * (i8 / ne)), e0 = TN * (i8 % ne);
    if (t0 >= T) return;
    uint8_t* const st = smem + wave * 2 * STAGE;
    const uint32_t c0 = wave * (hidden / 8), nc = hidden / 256;   // first column, chunks
    // load i: rows 8 i + lane / 8 (tokens, then experts), piece (lane % 8) ^ (row % 8);
    // rows past the last are the last
    const float* src[NL];
#pragma unroll
    for (uint32_t i = 0; i < NL; i++) {
        const uint32_t r = 8 * i + lane / 8;
        const float* row = 8 * i < TM ? x + (size_t)min(t0 + r, T - 1) * hidden
                                      : router + (size_t)min(e0 + r - TM, n_experts - 1) * hidden;
        src[i] = row + c0 + 4 * ((lane & 7u) ^ (r & 7u));
    }
    auto stage = [&](uint32_t c) {
#pragma unroll
        for (uint32_t i = 0; i < NL; i++)
            __builtin_amdgcn_global_load_lds((glb_void_t*)(src[i] + 32 * c), (lds_void_t*)(st + (c & 1u) * STAGE + 1024 * i),
                                             16, 0, 0);
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 sum[MM][NN];   // of the chunks so far
#pragma unroll
    for (int i = 0; i < MM; i++)
#pragma unroll
        for (int j = 0; j < NN; j++) sum[i][j] = zero;
    stage(0);
    if (nc > 1) stage(1);
    for (uint32_t c = 0; c < nc; c++) {
        // chunk c has landed (vmcnt: only the next one's NL loads may be in flight)
        if (c + 1 < nc) __builtin_amdgcn_s_waitcnt(0x0f70u | NL);
        else __builtin_amdgcn_s_waitcnt(0x0f70u);
        const uint8_t* s = st + (c & 1u) * STAGE + 128 * m;
        f32x4 a[2][MM], b[2][NN];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t o = 16 * ((4 * h + g) ^ (m & 7u));
#pragma unroll
            for (int i = 0; i < MM; i++) a[h][i] = *(const f32x4*)(s + 2048 * i + o);
#pragma unroll
            for (int j = 0; j < NN; j++) b[h][j] = *(const f32x4*)(s + 2048 * (MM + j) + o);
        }
        __builtin_amdgcn_s_waitcnt(0xc07fu);   // lgkmcnt(0): the chunk is in registers, its stage free
        __builtin_amdgcn_sched_barrier(0);
        if (c + 2 < nc) stage(c + 2);
#pragma unroll
        for (int i = 0; i < MM; i++)
#pragma unroll
            for (int j = 0; j < NN; j++) {
                f32x4 p[8];
#pragma unroll
                for (int k = 0; k < 8; k++)
                    p[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[k / 4][i][k % 4], b[k / 4][j][k % 4], zero, 0, 0, 0);
                sum[i][j] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            }
    }
    // the waves' sums through LDS, in their own stages: lane holds tokens 16 i + 4 g + q
    // of expert 16 j + m
    float* const red = (float*)smem;
    constexpr uint32_t WS = 2 * STAGE / 4;   // floats from wave to wave
    static_assert(TM * TN * 4 <= 2 * STAGE, "a wave's sums fit its stages");
#pragma unroll
    for (int i = 0; i < MM; i++)
#pragma unroll
        for (int j = 0; j < NN; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                red[wave * WS + (16 * i + 4 * g + q) * TN + 16 * j + m] = sum[i][j][q];
    __syncthreads();
    for (uint32_t o = tid; o < TM * TN; o += 512) {
        const uint32_t t = t0 + o / TN, e = e0 + o % TN;
        float v[8];
#pragma unroll
        for (int w = 0; w < 8; w++) v[w] = red[w * WS + o];
        if (t < T && e < n_experts)
            logits[(size_t)t * n_experts + e] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
}

template <int TM, int TN>
void launch_router(const PrefillLayer& L, const float* x, float* logits, hipStream_t st) {
    const uint32_t tt = (L.T + TM - 1) / TM, ne = (L.n_experts + TN - 1) / TN;
    k_pre_router_mfma<TM, TN><<<8 * ((tt + 7) / 8) * ne, 512, 0, st>>>(L.router, x, logits, L.hidden, L.n_experts, L.T);
}

// Router logits of T tokens: block (expert e, tokens 4c .. 4c+3), one wave.
// NV = hidden / 256 float4 per lane, a template constant, so the router row
// and the four tokens' inputs are requested at once (one memory round trip).
template <int NV>
__global__ __launch_bounds__(64) void k_pre_router(const float* __restrict__ router,
                                                   const float* __restrict__ x, float* logits,
                                                   uint32_t n_experts, uint32_t T) {
    constexpr uint32_t hidden = 256 * NV;
    const uint32_t e = blockIdx.x, t0 = 4 * blockIdx.y, lane = threadIdx.x;
    const float4* wr = (const float4*)(router + (size_t)e * hidden);
    float4 w[NV], xv[4][NV];
#pragma unroll
    for (int i = 0; i < NV; i++) w[i] = wr[64 * i + lane];
#pragma unroll
    for (uint32_t t = 0; t < 4; t++) {
        const float4* xr = (const float4*)(x + (size_t)min(t0 + t, T - 1) * hidden);
#pragma unroll
        for (int i = 0; i < NV; i++) xv[t][i] = xr[64 * i + lane];
    }
#pragma unroll
    for (uint32_t t = 0; t < 4; t++) {
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            acc = fmaf(w[i].x, xv[t][i].x, acc); acc = fmaf(w[i].y, xv[t][i].y, acc);
            acc = fmaf(w[i].z, xv[t][i].z, acc); acc = fmaf(w[i].w, xv[t][i].w, acc);
        }
        const float v = group_sum<64>(acc);
        if (lane == 0 && t0 + t < T) logits[(size_t)(t0 + t) * n_experts + e] = v;
    }
}

// Launch one matrix kind (formats fmask).
template <int MODE>
int launch_gemm(uint32_t fmask, const PrefillLayer& L, const PrefillWs& ws, hipStream_t st) {
    uint32_t lds = 0;
    for (int f = 0; f < F_NFMT; f++)
        if ((fmask >> f) & 1u) lds = lds > gemm_lds<MODE>(f, L.inter) ? lds : gemm_lds<MODE>(f, L.inter);
    // tiles of an XCD at most: an eighth of each kind, rounded up
    const uint32_t per = prefill_tiles_max(L.T, L.top_k, L.n_experts, L.three) / 8 + 2;
    const uint32_t grid = 8 * per * gemm_row_blocks<MODE>(L.hidden, L.inter);
    if (L.three) k_pre_gemm<MODE, 3><<<grid, 64 * kGW, lds, st>>>(L, ws);
    else k_pre_gemm<MODE, 2><<<grid, 64 * kGW, lds, st>>>(L, ws);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return qw6_fail("batched kernel launch: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace

bool prefill_supports(int f) { return f >= F_Q4K && f <= F_IQ3S; }

int prefill_forward(const PrefillLayer& L, const PrefillWs& ws, hipStream_t st) {
    if (L.hidden % 256 || L.inter % 256)
        return qw6_fail("batched path needs hidden, inter multiples of 256");
    const uint32_t all = (1u << F_NFMT) - 1u;
    if (!L.fmask_gu || !L.fmask_dn || (L.fmask_gu & ~all) || (L.fmask_dn & ~all) ||
        (L.sg.p && (!prefill_supports(L.sg.fmt) || !prefill_supports(L.sd.fmt) ||
                    L.su.fmt != L.sg.fmt)))
        return qw6_fail("batched path: unsupported expert format");
    if (L.top_k == 0 || L.top_k > 8 || L.n_experts > 256)
        return qw6_fail("batched path: top_k / n_experts out of range");
    if (L.hidden > 8 * kPWG) return qw6_fail("batched path needs hidden <= %u", 8 * kPWG);
    const float* logits = L.logits;
    const bool xn = !logits && L.norm_w;   // the router reads the norm that k_pre_x forms
    if (xn) k_pre_x<false><<<L.T, kPWG, 0, st>>>(L, ws, nullptr);
    if (!logits) {
        const float* xin = xn ? ws.xn : L.x;
        // One wave per expert and four tokens up to 10240 logits (256 experts, hidden
        // 2048, us: 33 tokens 5.6, 64 tokens 8.1; the matrix kernel 6.1 and 6.1: its
        // workgroups take a whole tile's time however few they are). Then tiles of
        // 16 x 16 up to two workgroups per CU, 32 x 32 beyond, which read half as much
        // per product (512 tokens 10.6 and 15.7, 1024: 18.9 and 16.9, 2048: 35.9 and 32.0).
        // Over 16 to 256 experts, hidden 256 to 2048 and 17 to 2048 tokens the choice is never
        // slower than a wave per expert throughout, and within 1.2 times the fastest of the
        // three but for 16 experts at 640 tokens (9.0 us, the 16 x 16 tiles 5.4).
        const uint32_t nv = L.hidden / 256, nl = L.T * L.n_experts;
        const dim3 g(L.n_experts, (L.T + 3) / 4);
        if (nv != 1 && nv != 2 && nv != 4 && nv != 8)
            return qw6_fail("batched router needs hidden in {256, 512, 1024, 2048}");
        if (nl > 512 * 256) launch_router<32, 32>(L, xin, ws.logits, st);
        else if (nl > 10240) launch_router<16, 16>(L, xin, ws.logits, st);
        else if (nv == 1) k_pre_router<1><<<g, 64, 0, st>>>(L.router, xin, ws.logits, L.n_experts, L.T);
        else if (nv == 2) k_pre_router<2><<<g, 64, 0, st>>>(L.router, xin, ws.logits, L.n_experts, L.T);
        else if (nv == 4) k_pre_router<4><<<g, 64, 0, st>>>(L.router, xin, ws.logits, L.n_experts, L.T);
        else k_pre_router<8><<<g, 64, 0, st>>>(L.router, xin, ws.logits, L.n_experts, L.T);
        logits = ws.logits;
    }
    if (xn) k_pre_route<<<L.T, 64, 0, st>>>(L, ws, logits);
    else k_pre_x<true><<<L.T, kPWG, 0, st>>>(L, ws, logits);
    k_pre_sort<<<1, 1024, 0, st>>>(L, ws);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return qw6_fail("batched routing launch: %s", hipGetErrorString(e));
    if (launch_gemm<0>(L.fmask_gu | (L.sg.p ? 1u << L.sg.fmt : 0u), L, ws, st)) return -1;
    if (launch_gemm<1>(L.fmask_dn | (L.sg.p ? 1u << L.sd.fmt : 0u), L, ws, st)) return -1;
    k_pre_combine<<<dim3(L.T, (L.hidden / 4 + 255) / 256), 256, 0, st>>>(L, ws);
    e = hipGetLastError();
    if (e != hipSuccess) return qw6_fail("batched combine launch: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace qw6
