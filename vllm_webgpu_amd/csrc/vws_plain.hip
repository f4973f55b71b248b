// vws_plain.hip -- sampling launches whose rows nothing cuts: temperature alone (no top-k, top-p or
// min-p arrays), no processors, penalties, mask, soft cap or logprobs, in one read of the logits;
// and all-greedy launches of the same kind where rows outnumber the compute units or fill at
// most half of them (400 x 32000 fp32: 35 us with one row per compute unit -> 10.8 us).
//
// A row's token is the largest exponential-race key e_i / (-ln u_i), e_i = exp_det(y_i - max y).
// The keys' bits need the row maximum, but their order hardly does: with E = -ln u,
//     log2 key_i = x_i c - log2 E_i - const,  c = log2(e) / T,
// so each part of a row keeps the elements whose g_i = x_i c - log2 E_i lies within delta of the
// largest seen (a handful), delta a bound on the rounding of both forms, and the part that
// arrives last computes the exact keys of those alone, with the row maximum known.  It reads the
// row again (exact_row) only when the short lists cannot decide it: no finite maximum, or one
// whose x c is at the edge of fp32's range, uniforms outside [0, 1), more near-equal keys than a
// list holds, a best key near underflow, an infinite temperature.
//
// Bound: VALU, by the generated uniforms (Philox-4x32-10: 20 quarter-rate 32 x 32 multiplies per
// four tokens).  E >= 1 - u >= 2^-24 gives each block of four tokens the bound max x c + 24, so
// the blocks that cannot win are dropped first and the others are queued per wave until 64 of
// them fill its lanes; per token one hardware log2 of 1 - u (E >= 1 - u: an upper bound of g)
// decides whether log_det and the second log2 are computed at all.  128 rows of 151936 bf16
// logits: 257 us on the multi-pass path (one workgroup per row, three transcendental sequences
// and a division per element) -> 30.3 us; 4 rows 244 -> 11.6 us; 256 rows of fp32 with given uniforms
// (read whole: 311 MB) 227 -> 55 us.
#include "vws_plain.h"

namespace vws {

constexpr int kPlWaves = kPlThreads / kWave;
constexpr int kPlQueue = 2 * kWave;      // queued blocks per wave
constexpr int kPlCand = 256;             // candidates listed per part
constexpr int kPlBlocks = 2;             // blocks of four tokens per lane and iteration

struct PlainSmem {
    alignas(16) float4 qx[kPlWaves][kPlQueue];   // queued blocks: their logits
    uint32_t qb[kPlWaves][kPlQueue];             // and block numbers
    alignas(16) uint64_t recs[kPlMaxParts][8];   // the parts' records (own first)
    uint32_t cidx[kPlCand];                      // candidates: token, logit, g
    float cx[kPlCand], cg[kPlCand];
    uint32_t ncand, nsel, bad, thr, last;
    uint32_t maxk;
    uint32_t count;
    uint64_t red[kPlWaves][3];
};

__shared__ PlainSmem g_plain_sh;

// A part's record: words 0 (largest key << 32 | NaN elements), 1 (candidates, or
// kPlOver) and 2-7 (candidates: token << 32 | logit bits).  Greedy rows: word 0 the best
// (key << 32 | 0x7FFFFFFF - index).
constexpr uint32_t kPlOver = 0xFFFFFFFFu;

// The four logits of block b: one 16- or 8-byte load at the element's own alignment (rows of
// 16-bit logits that start on an odd element are read one by one).
template <typename T>
struct Block4;
template <>
struct Block4<float> {
    static __device__ __forceinline__ float4 load(__amdgpu_buffer_rsrc_t rs, uint32_t b, bool) {
        const auto w = __builtin_amdgcn_raw_buffer_load_b128(rs, 16u * b, 0u, 2 /* nt */);
        return make_float4(u2f((uint32_t)w[0]), u2f((uint32_t)w[1]), u2f((uint32_t)w[2]), u2f((uint32_t)w[3]));
    }
};
template <typename T>
struct Block4 {
    static __device__ __forceinline__ float4 load(__amdgpu_buffer_rsrc_t rs, uint32_t b, bool dword) {
        uint32_t w0, w1;
        if (dword) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b64(rs, 8u * b, 0u, 2 /* nt */);
            w0 = (uint32_t)w[0];
            w1 = (uint32_t)w[1];
        } else {
            const uint32_t h0 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 8u * b, 0u, 0);
            const uint32_t h1 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 8u * b + 2u, 0u, 0);
            const uint32_t h2 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 8u * b + 4u, 0u, 0);
            const uint32_t h3 = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, 8u * b + 6u, 0u, 0);
            w0 = h0 | (h1 << 16);
            w1 = h2 | (h3 << 16);
        }
        float v[8];
        Elem<T>::from_words(w0, w1, 0u, 0u, v);
        return make_float4(v[0], v[1], v[2], v[3]);
    }
};

__device__ __forceinline__ float plain_uniform(const PlainArgs& a, int r, int t) {
    if (a.u) return a.u[(size_t)r * a.ustride + t];
    return philox_uniform(a.rng_seed ? a.rng_seed[r] : a.rng_key,
                          a.rng_seed ? (a.rng_offset ? a.rng_offset[r] : 0ull) : (uint64_t)(uint32_t)r,
                          (uint32_t)t);
}

// delta: g values this close may order differently as exact keys.  For elements that can win,
// |x c| <= |thr| + 31 (log2 E lies in [-24, 7]); the two forms differ by the roundings of x c (3
// of |x c|), y = x / T and y - max (1 each), by exp_det (1 ulp) and by the hardware log2 (1 ulp of
// at most 24: 2^-19); twice that, and the near-tie flag's 1e-6, is below
// 2^-16 + 2^-20 (|thr| + 64).
__device__ __forceinline__ float plain_delta(float thr) {
    return 0x1p-16f + 0x1p-20f * (__builtin_fabsf(thr) + 64.0f);
}

__device__ __forceinline__ float wave_max_f32(float v) {  // (no NaN)
    return val_of(wave_max_u32(key_of(v)));
}

// Writes row r's result (thread 0's race totals).
__device__ __forceinline__ void plain_write(const PlainArgs& a, int r, int32_t tok, uint32_t fl, int32_t kept) {
    a.sampled[r] = tok;
    if (a.flags) a.flags[r] = fl;
    if (a.nkept) a.nkept[r] = kept;
}
__device__ __forceinline__ uint32_t plain_near_tie(const RowRace& rs) {
    if (!rs.best || !rs.second) return 0u;
    const float bk = u2f((uint32_t)(rs.best >> 32)), sk = u2f(rs.second - 1u);
    return (double)sk >= (double)bk * (1.0 - 1e-6) ? VWS_FLAG_RACE_NEAR_TIE : 0u;
}

// rs merged over the workgroup, valid in thread 0 (two barriers).
__device__ __forceinline__ void plain_merge(PlainSmem& sm, RowRace& rs) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    rs.shfl_merge(32); rs.shfl_merge(16); rs.shfl_merge(8);
    rs.shfl_merge(4); rs.shfl_merge(2); rs.shfl_merge(1);
    __syncthreads();
    if (lane == 0) {
        sm.red[wave][0] = rs.best;
        sm.red[wave][1] = rs.last;
        sm.red[wave][2] = ((uint64_t)rs.second << 32) | rs.nkept;
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int w = 1; w < kPlWaves; ++w) {
            RowRace o;
            o.best = sm.red[w][0];
            o.last = sm.red[w][1];
            o.second = (uint32_t)(sm.red[w][2] >> 32);
            o.nkept = (uint32_t)sm.red[w][2];
            rs.merge(o);
        }
    }
}

// A row the lists cannot decide, by one workgroup: the row maximum is maxk; the best exact key (or,
// without a finite maximum, the first index of the largest key of y).  Only rows without a
// finite maximum, with uniforms outside [0, 1) or with very many near-equal keys come here in
// earnest.
//
// One workgroup reads the row again, so it is bound by the latency of its loads (EX blocks per lane,
// twice, in flight) and, where the keys decide, by their arithmetic: once an exact key of at
// least 2^-91 is known (see plain_kernel), an element whose bound of g (E >= 1 - u, and before the
// uniforms are generated E >= 2^-24) is below that key's g and delta is not computed; one whose
// uniform is outside [0, 1), which the bound does not hold for, always is.  Reading one element per
// load and computing every key it took 128 rows of 151936 bf16 logits with a +inf 343 us (55 now)
// and 128 of 128256 fp32 with a uniform of 1 each 587 us (152 now; the multi-pass path 85 and 158).
//
// A function of its own (which reads the kernel's arguments again), so that its registers and code
// stay out of the kernel: 128 rows of 151936 bf16 logits none of which comes here 32.9 -> 30.3 us,
// 256 x 151936 fp32 with given uniforms 55.1 -> 55.2.
template <typename T>
__device__ __noinline__ void exact_row(uint64_t kernarg, int r, uint32_t maxk) {
#if defined(__HIP_DEVICE_COMPILE__)
    using ArgsConst = const PlainArgs __attribute__((address_space(4)));
    const uint64_t ka = ((uint64_t)tp_first((uint32_t)(kernarg >> 32)) << 32) | tp_first((uint32_t)kernarg);
    const PlainArgs a = *(ArgsConst*)ka;
    r = (int)tp_first((uint32_t)r);
    maxk = tp_first(maxk);
    PlainSmem& sm = g_plain_sh;
    const T* row = reinterpret_cast<const T*>(a.logits) + (size_t)r * a.lstride;
    const float Tt = a.temperature[r];  // (no greedy row comes here)
    const float c = kPlLog2e / Tt;
    const int tid = threadIdx.x, lane = tid & 63;
    constexpr int EX = sizeof(T) == 4 ? 4 : 8;  // (8 of fp32 would leave the kernel two workgroups a CU)
    const int nblk = a.V >> 2;
    const int nit = (nblk + kPlThreads * EX - 1) / (kPlThreads * EX);
    const bool dword = (reinterpret_cast<uintptr_t>(row) & 3u) == 0u;
    const bool gen = a.u == nullptr;
    const float inf = __builtin_inff();
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(row, (uint32_t)nblk * 4u * (uint32_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t us = make_rsrc(gen ? (const void*)row : (const void*)(a.u + (size_t)r * a.ustride),
                                                gen ? 0u : (uint32_t)nblk * 16u);
    if (tid == 0) sm.thr = 0u;
    __syncthreads();
    // f(x, t, ok) for every four tokens t .. t + 3, ascending in a lane: the row's blocks (ok: of
    // the row), then the V % 4 tokens past them, the others NaN.  A wave goes on while f is true.
    auto blocks = [&](auto f) __attribute__((always_inline)) {
        float4 X[EX], Y[EX];
        auto load = [&](float4 (&d)[EX], int it) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < EX; ++q)
                d[q] = Block4<T>::load(rs, (uint32_t)((it * EX + q) * kPlThreads + tid), dword);
        };
        load(X, 0);
        for (int it = 0; it < nit; ++it) {
            load(Y, it + 1);
#pragma unroll
            for (int q = 0; q < EX; ++q) {
                const int b = (it * EX + q) * kPlThreads + tid;
                const float x[4] = {X[q].x, X[q].y, X[q].z, X[q].w};
                if (!f(x, 4 * b, b < nblk)) return;
            }
#pragma unroll
            for (int q = 0; q < EX; ++q) X[q] = Y[q];
        }
        if (tid < kWave && (a.V & 3)) {
            const int t0 = nblk << 2;
            float x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                x[j] = lane == 0 && t0 + j < a.V ? Elem<T>::load1(row + t0 + j) : __builtin_nanf("");
            f(x, t0, lane == 0);
        }
    };
    float m = maxk ? val_of(maxk) / Tt : __builtin_nanf("");
    RowRace rr;
    if (Tt == inf) {
        // y is 0 for a finite logit and NaN for an infinite one, the largest among them
        int any = 0;
        blocks([&](const float (&x)[4], int, bool ok) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 4; ++j) any |= ok && __builtin_fabsf(x[j]) < inf ? 1 : 0;
            return wave_ballot(any != 0) == 0ull;
        });
        m = __syncthreads_or(any) ? 0.0f : __builtin_nanf("");
    }
    if (!(m > -inf && m < inf)) {
        // the first token whose y is m: every y is NaN then (token 0), or every other one is
        // -inf, or (y has overflowed) x c has nearly too
        if (m == m)
            blocks([&](const float (&x)[4], int t, bool ok) __attribute__((always_inline)) {
                bool in[4], any = false;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    in[j] = ok && rr.best == 0ull && (m < 0.0f ? x[j] == x[j] : x[j] * c >= 0x1p127f);
                    any = any || in[j];
                }
                if (wave_ballot(any) != 0ull) {
#pragma unroll
                    for (int j = 3; j >= 0; --j)  // (the lowest index has the largest, and is the lane's first)
                        rr.best = in[j] && x[j] / Tt == m ? 0x7FFFFFFFull - (uint32_t)(t + j) : rr.best;
                    if (rr.best) atomicMax(&sm.thr, (uint32_t)rr.best);
                }
                // (what follows in this wave lies past its first lane's tokens)
                const uint32_t first = __hip_atomic_load(&sm.thr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                return tp_first(first) <= 0x7FFFFFFFu - tp_first((uint32_t)t);
            });
        plain_merge(sm, rr);
        if (tid == 0) plain_write(a, r, rr.best ? (int32_t)(0x7FFFFFFFu - (uint32_t)rr.best) : 0, VWS_FLAG_DEGENERATE, 1);
        return;
    }
    // whether g orders this row's keys (see plain_kernel)
    const bool ordered = Tt < inf && __builtin_fabsf(val_of(maxk) * c) < 0x1p127f;
    const uint64_t seed = gen ? (a.rng_seed ? a.rng_seed[r] : a.rng_key) : 0ull;
    const uint64_t off = a.rng_seed ? (a.rng_offset ? a.rng_offset[r] : 0ull) : (uint64_t)(uint32_t)r;
    float thr = -inf, lim = -inf;  // (wave-uniform)
    blocks([&](const float (&x)[4], int t, bool ok) __attribute__((always_inline)) {
        const float bm = __builtin_fmaxf(__builtin_fmaxf(x[0], x[1]), __builtin_fmaxf(x[2], x[3]));
        bool in[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            in[j] = ok && x[j] == x[j] && (Tt < inf || __builtin_fabsf(x[j]) < inf);  // (y is not NaN)
            rr.nkept += in[j] ? 1u : 0u;
        }
        if (gen && wave_ballot(ok && !(__builtin_fmaf(bm, c, 24.0f) < lim)) == 0ull) return true;
        float u[4];
        if (gen) {
            uint32_t k[4] = {(uint32_t)t >> 2, (uint32_t)off, (uint32_t)(off >> 32), 0u};
            philox4x32_10(k, (uint32_t)seed, (uint32_t)(seed >> 32));
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = philox_word_uniform(k[j]);
        } else if (t + 4 <= a.V) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b128(us, 4u * (uint32_t)t, 0u, 2);
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = u2f((uint32_t)w[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) u[j] = in[j] ? plain_uniform(a, r, t + j) : 0.5f;
        }
        bool need[4], any = false;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float z = __builtin_fmaf(x[j], c, -__builtin_amdgcn_logf(1.0f - u[j]));
            need[j] = in[j] && !(u[j] >= 0.0f && u[j] < 1.0f && z < lim);
            any = any || need[j];
        }
        if (wave_ballot(any) == 0ull) return true;
        float top = -inf;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (!need[j]) continue;
            const float y = x[j] / Tt;
            const uint64_t lk = ((uint64_t)key_of(y) << 32) | (uint32_t)(t + j);
            rr.last = rr.last > lk ? rr.last : lk;
            const float E = 0.0f - log_det(u[j]);
            const float key = exp_det(y - m) / E;
            rr.add_key(key, t + j);
            if (u[j] < 1.0f && key >= 0x1p-91f) top = __builtin_fmaxf(top, __builtin_fmaf(x[j], c, -__builtin_amdgcn_logf(E)));
        }
        if (!ordered) return true;
        const uint32_t st = tp_first(__hip_atomic_load(&sm.thr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        if (st) thr = __builtin_fmaxf(thr, val_of(st));
        if (wave_ballot(top > thr)) {
            thr = wave_max_f32(__builtin_fmaxf(top, thr));
            if (lane == 0) atomicMax(&sm.thr, key_of(thr));
        }
        lim = thr - plain_delta(thr);
        return true;
    });
    plain_merge(sm, rr);
    if (tid == 0)
        plain_write(a, r, rr.best ? (int32_t)(0x7FFFFFFF - (uint32_t)rr.best) : (int32_t)(uint32_t)rr.last,
                    plain_near_tie(rr), (int32_t)rr.nkept);
#else
    (void)kernarg; (void)r; (void)maxk;
#endif
}

template <typename T>
__global__ __launch_bounds__(kPlThreads) void plain_kernel(PlainArgs a) {
#ifdef VWS_TRACE
    const uint64_t tr_entry = trace_clock();
#endif
    PlainSmem& sm = g_plain_sh;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = a.S;
    const int r = blockIdx.x / S, p = blockIdx.x - r * S;
    const T* row = reinterpret_cast<const T*>(a.logits) + (size_t)r * a.lstride;
    const float Tt = a.temperature ? a.temperature[r] : 0.0f;
    const bool greedy = is_greedy(Tt);
    const bool gen = a.u == nullptr;
    const uint64_t seed = gen ? (a.rng_seed ? a.rng_seed[r] : a.rng_key) : 0ull;
    const uint64_t off = a.rng_seed ? (a.rng_offset ? a.rng_offset[r] : 0ull) : (uint64_t)(uint32_t)r;
    const float* urow = gen ? nullptr : a.u + (size_t)r * a.ustride;
    auto traced = [&]() {  // trace build: the workgroup's record
#ifdef VWS_TRACE
        trace_mark(a, VWS_TRACE_ROW);
        trace_put(a, VWS_TRACE_ENTRY, tr_entry);
        trace_put(a, VWS_TRACE_XCC, trace_xcc());
        trace_put(a, VWS_TRACE_ROWID, (uint64_t)r);
        trace_mark(a, VWS_TRACE_EXIT);
#endif
    };
    // blocks of four tokens [b0, b1); the V % 4 tokens past the last block are thread 0's of the
    // last part
    const int nblk = a.V >> 2;
    const int b0 = p * a.part_blocks, b1 = min(nblk, b0 + a.part_blocks);
    const bool dword = (reinterpret_cast<uintptr_t>(row) & 3u) == 0u;
    // (the resources end with the part: what is asked for past it is zeros and not fetched)
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(row, (uint32_t)b1 * 4u * (uint32_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t us = make_rsrc(gen ? (const void*)row : (const void*)urow,
                                                gen ? 0u : (uint32_t)b1 * 16u);
    if (tid == 0) { sm.ncand = 0u; sm.nsel = 0u; sm.bad = 0u; sm.thr = 0u; sm.maxk = 0u; sm.count = 0u; }
    __syncthreads();

    const float c = kPlLog2e / (greedy ? 1.0f : Tt);
    float thr = -__builtin_inff();   // a lower bound of the part's largest g (wave-uniform)
    float mx = __builtin_nanf("");   // the lane's largest logit
    uint32_t nan = 0u;               // NaN elements (wave-uniform)
    float lim24 = -__builtin_inff(); // thr less its delta and 24 (see below)
    int bblk = b0 + tid;             // greedy rows: the first block that holds the lane's largest
    int nq = 0;                      // blocks queued (wave-uniform)
    bool bad = false;

    // Tokens t .. t + 3 with logits x and v = 1 - u (ok: a block of the row; v <= 1): the
    // candidates among them into the list, the wave's threshold raised.
    auto race4 = [&](const float (&x)[4], const float (&v)[4], const float (&u)[4], uint32_t t, bool ok)
        __attribute__((always_inline)) {
        float z[4], zm = -__builtin_inff(), lb = -__builtin_inff();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // E >= v: an upper bound of g; E <= 1.3863 v for v <= 1/2: a lower one 0.4713 below
            z[j] = __builtin_fmaf(x[j], c, -__builtin_amdgcn_logf(v[j]));
            z[j] = ok && z[j] == z[j] ? z[j] : -__builtin_inff();
            zm = __builtin_fmaxf(zm, z[j]);
            lb = v[j] <= 0.5f ? __builtin_fmaxf(lb, z[j] - 0.4720f) : lb;
        }
        if (wave_ballot(zm >= thr) == 0ull && wave_ballot(zm >= thr - plain_delta(thr)) == 0ull) return;
        {
            // other waves' threshold, and this step's lower bounds
            const uint32_t st = tp_first(__hip_atomic_load(&sm.thr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
            if (st) thr = __builtin_fmaxf(thr, val_of(st));
            lb -= plain_delta(lb);
            if (wave_ballot(lb > thr)) thr = wave_max_f32(__builtin_fmaxf(lb, thr));
        }
        float lim = thr - plain_delta(thr);
        float top = -__builtin_inff();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (!(z[j] >= lim) || z[j] == -__builtin_inff()) continue;
            const float E = 0.0f - log_det(u[j]);
            const float g = __builtin_fmaf(x[j], c, -__builtin_amdgcn_logf(E));
            if (!(g >= lim) || g == -__builtin_inff()) continue;
            top = __builtin_fmaxf(top, g);
            const uint32_t pos = atomicAdd(&sm.ncand, 1u);
            if (pos < (uint32_t)kPlCand) {
                sm.cidx[pos] = t + (uint32_t)j;
                sm.cx[pos] = x[j];
                sm.cg[pos] = g;
            }
        }
        if (wave_ballot(top > thr)) {
            thr = wave_max_f32(__builtin_fmaxf(top, thr));
            if (lane == 0) atomicMax(&sm.thr, key_of(thr));
        }
        lim24 = thr - plain_delta(thr) - 24.0f;
    };
    // the first n (<= 64) queued blocks, one per lane; the rest moves to the front
    auto drain = [&](int n) __attribute__((always_inline)) {
        const bool ok = lane < n;
        const float4 xq = sm.qx[wave][lane];
        const uint32_t b = sm.qb[wave][lane];
        const float4 xr = sm.qx[wave][lane + kWave];
        const uint32_t br = sm.qb[wave][lane + kWave];
        wave_sync();
        sm.qx[wave][lane] = xr;
        sm.qb[wave][lane] = br;
        wave_sync();
        nq -= n;
        uint32_t k[4] = {b, (uint32_t)off, (uint32_t)(off >> 32), 0u};
        philox4x32_10(k, (uint32_t)seed, (uint32_t)(seed >> 32));
        const float x[4] = {xq.x, xq.y, xq.z, xq.w};
        float v[4], u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            u[j] = philox_word_uniform(k[j]);
            v[j] = 1.0f - u[j];  // exact: u is a multiple of 2^-24
        }
        race4(x, v, u, 4u * b, ok);
    };

    const int nit = (b1 - b0 + kPlThreads * kPlBlocks - 1) / (kPlThreads * kPlBlocks);
    float4 X[kPlBlocks], Y[kPlBlocks];
    auto load = [&](float4 (&d)[kPlBlocks], int it) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < kPlBlocks; ++q)
            d[q] = Block4<T>::load(rs, (uint32_t)(b0 + (it * kPlBlocks + q) * kPlThreads + tid), dword);
    };
    load(X, 0);
    for (int it = 0; it < nit; ++it) {
        load(Y, it + 1);  // (past the part's blocks: zeros, nothing fetched)
#pragma unroll
        for (int q = 0; q < kPlBlocks; ++q) {
            const int b = b0 + (it * kPlBlocks + q) * kPlThreads + tid;
            const bool ok = b < b1;
            const float x[4] = {X[q].x, X[q].y, X[q].z, X[q].w};
            float bm = __builtin_fmaxf(__builtin_fmaxf(x[0], x[1]), __builtin_fmaxf(x[2], x[3]));
            bm = ok ? bm : __builtin_nanf("");
            if (!greedy &&
                (wave_ballot(__builtin_isunordered(x[0], x[1])) | wave_ballot(__builtin_isunordered(x[2], x[3])))) {
#pragma unroll
                for (int j = 0; j < 4; ++j) nan += (uint32_t)__popcll(wave_ballot(ok && x[j] != x[j]));
            }
            if (greedy) {
                // (ascending blocks: the first that reaches a value keeps it; mx is NaN at first)
                const bool up = bm > mx || (mx != mx && bm == bm);
                bblk = up ? b : bblk;
            }
            mx = __builtin_fmaxf(mx, bm);
            if (greedy) {
            } else if (gen) {
                // E >= 2^-24: no token of the block reaches max x c + 24 (NaN: no)
                const bool need = bm * c >= lim24;
                const uint64_t bal = wave_ballot(need);
                if (need) {
                    const int at = nq + lane_prefix(bal);
                    sm.qx[wave][at] = make_float4(x[0], x[1], x[2], x[3]);
                    sm.qb[wave][at] = (uint32_t)b;
                }
                nq += __popcll(bal);
                wave_sync();
                if (nq >= kWave) drain(kWave);
            } else {
                const auto w = __builtin_amdgcn_raw_buffer_load_b128(us, 16u * (uint32_t)b, 0u, 2);
                float v[4], u[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u[j] = u2f((uint32_t)w[j]);
                    bad = bad || (ok && !(u[j] >= 0.0f && u[j] < 1.0f));
                    v[j] = 1.0f - u[j];
                }
                race4(x, v, u, 4u * (uint32_t)b, ok);
            }
        }
#pragma unroll
        for (int q = 0; q < kPlBlocks; ++q) X[q] = Y[q];
    }
    if (nq > 0) drain(nq);
    uint64_t gbest = 0ull;  // greedy rows: the largest key, the lowest index
    if (greedy && mx == mx) {
        const uint32_t km = key_of(mx);
#pragma unroll
        for (int j = 3; j >= 0; --j) {
            const int t = 4 * bblk + j;
            if (key_of(Elem<T>::load1(row + t)) == km) gbest = ((uint64_t)km << 32) | (uint32_t)(0x7FFFFFFF - t);
        }
    }
    // the tokens past the last block, by the first wave of the last part
    if (p == S - 1 && wave == 0 && (a.V & 3)) {
        const int t0 = nblk << 2;
        float x[4], v[4], u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool in = lane == 0 && t0 + j < a.V;
            x[j] = in ? Elem<T>::load1(row + t0 + j) : __builtin_nanf("");
            u[j] = in && !greedy ? plain_uniform(a, r, t0 + j) : 0.5f;
            v[j] = 1.0f - u[j];
            bad = bad || !(u[j] >= 0.0f && u[j] < 1.0f);
            nan += (uint32_t)__popcll(wave_ballot(in && x[j] != x[j]));
            mx = __builtin_fmaxf(mx, x[j]);
            const uint64_t pk = ((uint64_t)key_of(x[j]) << 32) | (uint32_t)(0x7FFFFFFF - (t0 + j));
            gbest = lane == 0 && t0 + j < a.V && pk > gbest ? pk : gbest;
        }
        if (!greedy) race4(x, v, u, (uint32_t)t0, lane == 0);
    }

    VWS_TRACE_MARK(a, VWS_TRACE_STREAM);
    // the part's record
    const uint32_t wk = wave_max_u32(key_of(mx));
    const uint64_t wg = wave_max_u64(gbest);
    const bool wbad = wave_ballot(bad) != 0ull;
    if (lane == 0) {
        atomicMax(&sm.maxk, wk);
        if (nan) atomicAdd(&sm.count, nan);
        if (wbad) atomicOr(&sm.bad, 1u);
        sm.red[wave][0] = wg;
    }
    __syncthreads();
    const uint32_t nc = sm.ncand;
    if (!greedy && tid < (int)nc && tid < kPlCand) {
        const float best = val_of(sm.thr);
        if (sm.cg[tid] >= best - plain_delta(best)) {
            const uint32_t pos = atomicAdd(&sm.nsel, 1u);
            if (pos < 6u) sm.recs[0][2 + pos] = ((uint64_t)sm.cidx[tid] << 32) | f2u(sm.cx[tid]);
        }
    }
    __syncthreads();
    if (tid == 0) {
        if (greedy) {
            uint64_t best = 0ull;
            for (int w = 0; w < kPlWaves; ++w) best = best > sm.red[w][0] ? best : sm.red[w][0];
            sm.recs[0][0] = best;
            sm.recs[0][1] = 0ull;
        } else {
            const uint32_t n = sm.nsel;
            sm.recs[0][0] = ((uint64_t)sm.maxk << 32) | sm.count;  // (NaN elements)
            sm.recs[0][1] = (nc > (uint32_t)kPlCand || n > 6u || sm.bad) ? kPlOver : n;
        }
    }
    __syncthreads();
    if (S > 1) {
        // published; the part that arrives last reads them all
        uint64_t* rec = a.rec + (size_t)r * S * 8;
        if (tid < 8) ag_store64(rec + p * 8 + tid, sm.recs[0][tid]);
        stores_complete();
        __syncthreads();
        if (tid == 0) sm.last = ag_add32(&a.ctr[r], 1u) == (uint32_t)(S - 1) ? 1u : 0u;
        __syncthreads();
        if (!sm.last) {
            traced();
            return;
        }
        if (tid == 0) ag_store32(&a.ctr[r], 0u);
        for (int i = tid; i < S * 8; i += kPlThreads) sm.recs[i >> 3][i & 7] = ag_load64(rec + i);
        __syncthreads();
    }
    // every thread: the row's totals (S <= 32)
    if (greedy) {
        if (tid == 0) {
            uint64_t best = 0ull;
            for (int i = 0; i < S; ++i) best = best > sm.recs[i][0] ? best : sm.recs[i][0];
            const bool any = (best >> 32) != 0ull;  // (an element that is not NaN)
            plain_write(a, r, any ? (int32_t)(0x7FFFFFFFu - (uint32_t)best) : 0, VWS_FLAG_GREEDY, 1);
        }
        traced();
        return;
    }
    uint32_t maxk = 0u, count = 0u, over = 0u, ntot = 0u;
    {
        const uint64_t w0 = lane < S ? sm.recs[lane][0] : 0ull;
        const uint32_t n = lane < S ? (uint32_t)sm.recs[lane][1] : 0u;
        maxk = wave_max_u32((uint32_t)(w0 >> 32));
        count = (uint32_t)a.V - (uint32_t)wave_sum_u64((uint32_t)w0);
        over = wave_ballot(n == kPlOver) != 0ull ? 1u : 0u;
        ntot = over ? 0u : (uint32_t)wave_sum_u64(n);
    }
    const float m = maxk ? val_of(maxk) / Tt : __builtin_nanf("");
    const bool fin = m > -__builtin_inff() && m < __builtin_inff();
    // x c of the largest logits at the edge of fp32's range: it can be infinite for one of two
    // neighbours that y holds equal, and g orders nothing there
    const bool past = !(__builtin_fabsf(val_of(maxk) * c) < 0x1p127f);
    // (an infinite temperature turns infinite logits into NaN, which the counts above miss)
    bool exact = !fin || past || over || ntot == 0u || Tt == __builtin_inff();  // (uniform)
    if (!exact) {
        // exact keys of the listed candidates (6 slots a part)
        RowRace rr;
        for (int i = tid; i < S * 6; i += kPlThreads) {
            const int q = i / 6, j = i - q * 6;
            if (j >= (int)(uint32_t)sm.recs[q][1]) continue;
            const uint64_t e = sm.recs[q][2 + j];
            const int t = (int)(uint32_t)(e >> 32);
            const float y = u2f((uint32_t)e) / Tt;
            rr.add_key(exp_det(y - m) / (0.0f - log_det(plain_uniform(a, r, t))), t);
        }
        plain_merge(sm, rr);
        // A key below 2^-91 decides nothing: exp_det is 0 below -80, so an element whose exact key is
        // 0 can have g only 80 log2(e) - 24 = 91.4 below the row maximum's x c (E >= 2^-24), and hide
        // a better live one of its part (where the largest logits drew u = 0).  From 2^-91 on no
        // exponential in reach is 0 and g orders the keys.
        const bool won = u2f((uint32_t)(rr.best >> 32)) >= 0x1p-91f;
        if (tid == 0) sm.last = won ? 1u : 0u;
        if (tid == 0 && won)
            plain_write(a, r, (int32_t)(0x7FFFFFFF - (uint32_t)rr.best), plain_near_tie(rr), (int32_t)count);
        __syncthreads();
        exact = !sm.last;
    }
#if defined(__HIP_DEVICE_COMPILE__)
    if (exact) exact_row<T>((uint64_t)__builtin_amdgcn_kernarg_segment_ptr(), r, maxk);
#endif
    traced();
}

template __global__ void plain_kernel<float>(PlainArgs);
template __global__ void plain_kernel<uint16_t>(PlainArgs);
template __global__ void plain_kernel<_Float16>(PlainArgs);

}  // namespace vws
