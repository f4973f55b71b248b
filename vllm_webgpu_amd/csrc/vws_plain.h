// vws_plain.h -- arguments of the kernel that samples rows nothing cuts (vws_plain.hip).
#pragma once

#include "vws_row.h"

namespace vws {

constexpr float kPlLog2e = 0x1.715476p+0f;  // log2(e) rounded to fp32

struct PlainArgs {
    const void* logits;
    int64_t lstride;
    int V;
    const float* temperature;    // null: every row greedy
    const float* u;              // [B, V] uniforms, or null: generated
    int64_t ustride;
    const uint64_t* rng_seed;
    const uint64_t* rng_offset;
    uint64_t rng_key;
    int32_t* sampled;
    uint32_t* flags;
    int32_t* nkept;
    int S;                       // parts per row (1: no workspace is used)
    int part_blocks;             // blocks of four tokens per part
    uint64_t* rec;               // [rows * S][8] (CoopState::plain_rec)
    uint32_t* ctr;               // [rows], left at zero
#ifdef VWS_TRACE
    uint64_t* trace;             // as KArgs::trace
    int trace_wgs;
#endif
};

__device__ __forceinline__ uint32_t tp_first(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

}  // namespace vws
