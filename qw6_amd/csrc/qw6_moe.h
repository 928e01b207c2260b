// qw6_moe.h -- types shared by the decode (qw6_hip.hip) and batched
// (qw6_prefill.hip) MoE FFN paths, and the batched path's host entry.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <type_traits>

namespace qw6 {

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) void glb_void_t;

// A load through a pointer to device global memory, emitted as a global
// load. A load through a generic pointer whose address space the compiler
// cannot infer (one read from memory, or a select of such pointers) is a
// FLAT load, which also counts in lgkmcnt: every later wait for an LDS
// operation then waits for it too, and a load issued ahead for the next
// step holds up the current step's LDS reads.
template <typename T>
__device__ __forceinline__ T ld_global(const void* p) {
    return *(const __attribute__((address_space(1))) T*)p;
}

// One weight matrix on the device (fmt: internal format, -1 = F32).
struct MatD {
    const uint8_t* p;
    int32_t fmt;
    uint32_t rows, cols, rb;   // rb: bytes per row
};

struct ExpertEnt {            // device expert table entry
    const uint8_t* p[3];      // gate, up, down
    int32_t fmt[3];
    uint32_t rb[3];
};

// Addressing of one matrix kind (gate / up / down) of the experts: a regular
// pack (expert e at base + e * stride, one format; the GGUF expert pack of
// bind_expert_pack, qw6.c:542-597) needs no memory round trip; otherwise the
// per-expert table entry is loaded.
struct PackRef {
    const uint8_t* base;
    uint64_t stride;
    int32_t fmt;
    uint32_t rb;
    uint32_t regular;
};

// Device workspace of the batched path, sized for max_tokens tokens.
struct PrefillWs {
    uint32_t* pidx;      // [T][top_k] selected experts
    float* pw;           // [T][top_k] gate weights
    uint32_t* ent_tok;   // [E] token of each entry (entries grouped by expert)
    float* ent_w;        // [E] gate weight of each entry
    uint32_t* ent_pos;   // [T][top_k] entry of (token, k)
    uint4* tiles;        // [n_tiles_max] {expert, first entry, count, 0}
    uint32_t* n_tiles;   // [2] tiles of more than 16 entries (first in the list), others
    float* logits;       // [T][n_experts]
    float* xn;           // [T][hidden] (RMSNorm of the input)
    uint16_t* xp;        // [T][hidden / 256][part][256] the input's two or three fp16 parts at
                         // the token's scale, columns in quad order (qw6_f16tile.h)
    uint2* xs;           // [T][hidden / 32] sums of those, three fp16 parts each
    float* xinv;         // [T] reciprocal of the token's scale
    uint16_t* mp;        // [E][inter / 256][part][256] the same of silu(gate) * up
    uint2* ms;           // [E][inter / 32]
    float* minv;         // [E][inter / 64] reciprocal scales of mid, one per 64 columns
    float* ybuf;         // [E][hidden]
};

struct PrefillLayer {
    uint32_t hidden, inter, n_experts, top_k, T;
    uint32_t three;               // activations in three parts, tiles of up to 16 entries (else two, 32)
    const float* x;
    const float* logits;          // given router logits or nullptr
    const float* router;          // F32 router or nullptr
    const float* shared_router;   // nullptr: shared weight 1
    const float* norm_w;          // RMSNorm weight or nullptr
    float norm_eps;
    const float* residual;
    float* out;
    uint32_t* idx_out;
    float* w_out;
    const ExpertEnt* experts;
    PackRef pk[3];
    uint32_t fmask_gu, fmask_dn;  // formats of the routed experts' gate/up (down): bit f
    MatD sg, su, sd;              // shared expert (sg.p == nullptr: none)
};

// Entries of a batch of T tokens: T * top_k routed, then T shared.
inline uint32_t prefill_entries(uint32_t T, uint32_t top_k) { return T * top_k + T; }
// Calls of fewer tokens hold the activations in three fp16 parts (24 bits, an fp32
// value within 2^38 of its group's largest), others in two (22 bits). The line is where
// the bf16 operands before them went from three parts (24 bits) to two (16), so that no
// call has less. Three parts cost most where tiles are full: 64 experts, 63 tokens 72 us,
// 64 tokens 63 us; over 256 experts nothing (117 and 114 us).
constexpr uint32_t kPrefill3PartBelow = 64;
// Entries per tile of the grouped kernels at most: two MFMA row groups of 16 that share one
// decoding of the weights, one where the activations take three parts.
__host__ __device__ constexpr uint32_t prefill_tile_entries(bool three) { return three ? 16u : 32u; }
// Tokens of one batch at most; longer calls run in batches of this many (the
// contraction's operand offsets are 32 bits: 2^16 rows of 2048 columns take 2^29 bytes).
constexpr uint32_t kPrefillMaxBatch = 65536;
// Tiles of a batch at most: the routed entries in tiles of one expert each
// (at most one partial tile per expert), then the shared expert's.
__host__ __device__ inline uint32_t prefill_tiles_max(uint32_t T, uint32_t top_k, uint32_t n_experts, bool three) {
    const uint32_t m = prefill_tile_entries(three);
    return (T * top_k + m - 1) / m + n_experts + (T + m - 1) / m;
}
// The workspace for calls of up to T tokens laid out from base (256-byte aligned);
// returns its bytes.
inline size_t carve_prefill_ws(uint8_t* base, uint32_t T, uint32_t hidden, uint32_t inter, PrefillWs* w) {
    constexpr uint32_t K8 = 8;   // top_k at most
    const size_t E = prefill_entries(T, K8);
    // the largest call in three parts
    const uint32_t T3 = T < kPrefill3PartBelow - 1 ? T : kPrefill3PartBelow - 1;
    const size_t E3 = prefill_entries(T3, K8);
    auto most = [](size_t a, size_t b) { return a > b ? a : b; };
    size_t o = 0;
    auto take = [&](auto*& p, size_t bytes) {
        p = base ? (std::remove_reference_t<decltype(p)>)(base + o) : nullptr;
        o += (bytes + 255) & ~(size_t)255;
    };
    PrefillWs d;
    take(d.pidx, (size_t)T * K8 * 4);
    take(d.pw, (size_t)T * K8 * 4);
    take(d.ent_tok, E * 4);
    take(d.ent_w, E * 4);
    take(d.ent_pos, (size_t)T * K8 * 4);
    take(d.tiles, most(prefill_tiles_max(T, K8, 256, false), prefill_tiles_max(T3, K8, 256, true)) * sizeof(uint4));
    take(d.n_tiles, 2 * 4);
    take(d.logits, (size_t)T * 256 * 4);
    take(d.xn, (size_t)T * hidden * 4);
    take(d.xp, most((size_t)T * 2, (size_t)T3 * 3) * hidden * 2);
    take(d.xs, (size_t)T * (hidden / 32) * 8);
    take(d.xinv, (size_t)T * 4);
    take(d.mp, most(E * 2, E3 * 3) * inter * 2);
    take(d.ms, E * (inter / 32) * 8);
    take(d.minv, E * (inter / 64) * 4);
    take(d.ybuf, E * hidden * 4);
    if (w) *w = d;
    return o;
}
// A workspace and the layer dimensions it holds (0 x 0: none yet).
struct PrefillWsOwner {
    PrefillWs ws;
    uint32_t hidden, inter;
};
// Make o hold a hidden x inter layer of T tokens (the same T on every call); alloc(bytes, &p):
// 0, or -1. The dimensions only grow, so layers of different shapes in turn
// allocate once; a failed allocation leaves o as it was. Every buffer comes from
// the one allocation, and the dimensions change with them or not at all. The
// allocation that a larger one replaces stays the context's until it is closed: a
// captured graph may hold its addresses (hidden and inter take four values each, so at
// most seven of them exist).
template <typename Alloc>
int grow_prefill_ws(PrefillWsOwner& o, uint32_t T, uint32_t hidden, uint32_t inter, Alloc alloc) {
    if (o.hidden >= hidden && o.inter >= inter) return 0;
    hidden = hidden > o.hidden ? hidden : o.hidden;
    inter = inter > o.inter ? inter : o.inter;
    void* p = nullptr;
    if (alloc(carve_prefill_ws(nullptr, T, hidden, inter, nullptr), &p)) return -1;
    carve_prefill_ws((uint8_t*)p, T, hidden, inter, &o.ws);
    o.hidden = hidden;
    o.inter = inter;
    return 0;
}
// Formats the grouped kernels decode (others take the per-token kernels).
bool prefill_supports(int fmt);
// Launch the batched MoE FFN on `st`; 0 or -1 (message via qw6_fail).
int prefill_forward(const PrefillLayer& L, const PrefillWs& ws, hipStream_t st);

int qw6_fail(const char* fmt, ...);

}  // namespace qw6
