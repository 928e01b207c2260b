// qw6_moe.h -- types shared by the decode (qw6_hip.hip) and batched
// (qw6_prefill.hip) MoE FFN paths, and the batched path's host entry.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

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
    uint16_t* xp;        // [T][hidden / 256][hi, lo][256] the input's fp16 parts at the
                         // token's scale, columns in quad order (qw6_f16tile.h)
    uint2* xs;           // [T][hidden / 32] sums of those, three fp16 parts each
    float* xinv;         // [T] reciprocal of the token's scale
    uint16_t* mp;        // [E][inter / 256][hi, lo][256] the same of silu(gate) * up
    uint2* ms;           // [E][inter / 32]
    float* minv;         // [E][inter / 64] reciprocal scales of mid, one per 64 columns
    float* ybuf;         // [E][hidden]
};

struct PrefillLayer {
    uint32_t hidden, inter, n_experts, top_k, T;
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
// Entries per tile of the grouped kernels at most (two MFMA row groups of 16
// that share one decoding of the weights).
constexpr uint32_t kPrefillTileEntries = 32;
// Tokens of one batch at most; longer calls run in batches of this many (the
// contraction's operand offsets are 32 bits: 2^16 rows of 2048 columns take 2^29 bytes).
constexpr uint32_t kPrefillMaxBatch = 65536;
// Tiles of a batch at most: the routed entries in tiles of one expert each
// (at most one partial tile per expert), then the shared expert's.
__host__ __device__ inline uint32_t prefill_tiles_max(uint32_t T, uint32_t top_k, uint32_t n_experts) {
    const uint32_t m = kPrefillTileEntries;
    return (T * top_k + m - 1) / m + n_experts + (T + m - 1) / m;
}
// Formats the grouped kernels decode (others take the per-token kernels).
bool prefill_supports(int fmt);
// Launch the batched MoE FFN on `st`; 0 or -1 (message via qw6_fail).
int prefill_forward(const PrefillLayer& L, const PrefillWs& ws, hipStream_t st);

int qw6_fail(const char* fmt, ...);

}  // namespace qw6
