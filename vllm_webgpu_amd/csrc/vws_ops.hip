// vws_ops.hip -- the standalone row operations of the library: batched argmax (the argmax.wgsl
// contract), row softmax with temperature (softmax.wgsl), in-place penalties, and the device
// self-test of the sampler arithmetic.
#include "vws_device.h"
#include "vws_internal.h"
#include "vws_sampler.h"

namespace vws {

constexpr int kOpThreads = 1024;
constexpr int kOpWaves = kOpThreads / 64;

__device__ __forceinline__ uint64_t op_block_max(uint64_t v, uint64_t* red) {
    v = wave_max_u64(v);
    __syncthreads();
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t t = 0;
#pragma unroll
    for (int i = 0; i < kOpWaves; ++i) t = t > red[i] ? t : red[i];
    return t;
}

__device__ __forceinline__ double op_block_sum_f64(double v, double* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    __syncthreads();
    if (lane_id() == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < kOpWaves; ++i) t += red[i];
    return t;
}

// One workgroup per row; (key << 32 | 0x7FFFFFFF - index) max = largest value, lowest index.
template <typename T>
__global__ __launch_bounds__(kOpThreads) void argmax_kernel(const T* logits, int64_t stride, int V,
                                                             int32_t* out) {
    __shared__ uint64_t red[kOpWaves];
    const int r = blockIdx.x;
    Slice<T> sl;
    sl.init(logits + (size_t)r * stride, 0, V);
    constexpr int VEC = Elem<T>::kVec;
    uint64_t best = 0;
    for (int c = threadIdx.x; c < sl.nchunks(); c += kOpThreads) {
        float v[VEC];
        const int i0 = sl.load(c, v);
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            const uint64_t pk = ((uint64_t)key_of(v[j]) << 32) | (uint32_t)(0x7FFFFFFF - (i0 + j));
            best = best > pk ? best : pk;
        }
    }
    best = op_block_max(best, red);
    if (threadIdx.x == 0) {
        int32_t tok = (int32_t)(0x7FFFFFFF - (uint32_t)(best & 0xFFFFFFFFu));
        if ((best >> 32) == 0u || tok >= V) tok = 0;  // every element NaN
        out[r] = tok;
    }
}

// probs = exp_det(x/T - m) / S, m = max x/T, S = sum exp_det(x/T - m), S in double.  Two forms,
// chosen by the launcher (vws_softmax):
//
// softmax_kernel, one workgroup per row (short rows, and calls whose probabilities overlap their
// logits): rows of up to 32 values per thread (V <= 32768 less the two unaligned edges) are read
// once and written once, each thread keeping its chunks in registers through the max, the sum
// and the write.  Longer rows are read twice: the maximum and S together (an online merge of
// per-thread running maxima and sums), then the write.
//
// softmax_part_kernel + softmax_write_kernel, several workgroups per row (any V): the first
// leaves each part's maximum and its sum relative to that maximum, the second combines a row's
// parts and writes the probabilities.  A row on one CU is bound by that CU's share of the
// bandwidth and by its issue slots (a division and two exponentials per element), so a batch
// smaller than the chip needs its rows split: 32 x 128256 fp32 95.5 -> 15.8 us.
//
// S is summed in another order than the sequential oracle (and, split, from rescaled partial
// sums); each probability is e * fl64(1 / S): the probabilities agree with the oracle's to
// within a few fp32 ulps.
template <typename T>
__global__ __launch_bounds__(kOpThreads) void softmax_kernel(const T* logits, int64_t stride, int V,
                                                              const float* temperature, float* probs,
                                                              float* row_max, float* log_sum) {
    __shared__ uint64_t red[kOpWaves];
    __shared__ double redd[kOpWaves];
    const int r = blockIdx.x;
    const float Tt = temperature ? temperature[r] : 1.0f;
    Slice<T> sl;
    sl.init(logits + (size_t)r * stride, 0, V);
    constexpr int VEC = Elem<T>::kVec;
    constexpr int kSoftmaxRegs = 32 / VEC;  // chunks a thread keeps in registers
    const int nch = sl.nchunks();
    // element i of chunk c (head and tail chunks are NaN-padded) lies in the row
    auto inside = [&](int c, int i) {
        const bool in = (c == 0) ? (i < sl.a) : (c <= sl.nbody ? true : i < V);
        return c <= sl.nbody + 1 && in && i < V;
    };
    float* out = probs + (size_t)r * V;
    uint64_t mk = 0;
    double s = 0.0;
    float m;
    double S;
    if (nch <= kSoftmaxRegs * kOpThreads) {
        // the row in registers: y = fl(x / T) once, then e = exp(y - m) in place of y, then
        // the probabilities e * fl64(1 / S) (within an ulp of e / S)
        float v[kSoftmaxRegs][VEC];
#pragma unroll
        for (int q = 0; q < kSoftmaxRegs; ++q) {
            const int c = threadIdx.x + q * kOpThreads;
            if (c < nch) {
                sl.load(c, v[q]);
            } else {
#pragma unroll
                for (int j = 0; j < VEC; ++j) v[q][j] = __builtin_nanf("");
            }
        }
        if (Tt != 1.0f) {
#pragma unroll
            for (int q = 0; q < kSoftmaxRegs; ++q)
#pragma unroll
                for (int j = 0; j < VEC; ++j) v[q][j] = v[q][j] / Tt;
        }
#pragma unroll
        for (int q = 0; q < kSoftmaxRegs; ++q)
#pragma unroll
            for (int j = 0; j < VEC; ++j) { const uint64_t k = key_of(v[q][j]); mk = mk > k ? mk : k; }
        mk = op_block_max(mk, red);
        m = mk ? val_of((uint32_t)mk) : -__builtin_inff();  // (a row of NaN: the empty maximum)
#pragma unroll
        for (int q = 0; q < kSoftmaxRegs; ++q)
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                // exp_det is 0 for NaN (NaN logits, padding, y - m of infinities)
                const float e = exp_det(v[q][j] - m);
                v[q][j] = e;
                const int c = threadIdx.x + q * kOpThreads;
                const int i0 = c == 0 ? 0 : sl.a + (c - 1) * VEC;
                if (c < nch && inside(c, i0 + j)) s += (double)e;
            }
        S = op_block_sum_f64(s, redd);
        const double inv = 1.0 / S;
#pragma unroll
        for (int q = 0; q < kSoftmaxRegs; ++q) {
            const int c = threadIdx.x + q * kOpThreads;
            // first element of chunk c: the row's start (head), the body vectors, the tail
            const int i0 = c == 0 ? 0 : sl.a + (c - 1) * VEC;
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (c < nch && inside(c, i0 + j)) out[i0 + j] = (float)((double)v[q][j] * inv);
        }
    } else {
        // longer rows: the maximum and the normaliser in one pass (each thread keeps a running
        // maximum mt of its finite values and its sum st of exp(y - mt), rescaled when mt
        // rises; the workgroup merges them as sum st * exp(mt - m)), then a second pass writes
        // the probabilities.  Only finite values add a term: exp_det is 0 for NaN, for -inf
        // and for y - m of infinities, so S is 0 when m is not finite.
        float mt = -__builtin_inff();
        double st = 0.0;
        for (int c = threadIdx.x; c < nch; c += kOpThreads) {
            float v[VEC];
            const int i0 = sl.load(c, v);
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                const float y = v[j] / Tt;
                const uint64_t k = key_of(y);
                mk = mk > k ? mk : k;
                if (!inside(c, i0 + j)) continue;  // padding of the head and tail chunks
                if (!(__builtin_fabsf(y) < __builtin_inff())) continue;
                if (y > mt) {
                    st = st * (double)exp_det(mt - y) + 1.0;
                    mt = y;
                } else {
                    st += (double)exp_det(y - mt);
                }
            }
        }
        mk = op_block_max(mk, red);
        m = mk ? val_of((uint32_t)mk) : -__builtin_inff();  // (a row of NaN: the empty maximum)
        const bool mfin = __builtin_fabsf(m) < __builtin_inff();
        S = op_block_sum_f64(mfin && mt > -__builtin_inff() ? st * (double)exp_det(mt - m) : 0.0, redd);
        const double inv = 1.0 / S;
        for (int c = threadIdx.x; c < nch; c += kOpThreads) {
            float v[VEC];
            const int i0 = sl.load(c, v);
#pragma unroll
            for (int j = 0; j < VEC; ++j)
                if (inside(c, i0 + j)) out[i0 + j] = (float)((double)exp_det(v[j] / Tt - m) * inv);
        }
    }
    if (threadIdx.x == 0) {
        if (row_max) row_max[r] = m;
        if (log_sum) log_sum[r] = (float)log(S);
    }
}

// ---- the split softmax -------------------------------------------------------------------

// A thread's elements of part p of a row, in registers: kPartVecs body vectors, then one edge
// element (the unaligned head and tail together hold fewer than 2 VEC elements, one per thread
// from thread 0 on).  Everything outside the part is NaN.
template <typename T>
struct SoftmaxPart {
    static constexpr int VEC = Elem<T>::kVec;
    static constexpr int kVecs = kSmPartMax / (kSmThreads * VEC);
    int lo, hi, a, nbody, edge;  // edge: this thread's edge element, or -1
    float v[kVecs][VEC];
    float ve;
    __device__ __forceinline__ void load(const T* row, int V, int part_len, int p, float Tt) {
        lo = p * part_len;
        hi = min(V, lo + part_len);
        Slice<T> sl;
        sl.init(row, lo, hi);
        a = sl.a;
        nbody = sl.nbody;
        const int tid = threadIdx.x;
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(row + a, 16u * (uint32_t)nbody);
#pragma unroll
        for (int q = 0; q < kVecs; ++q) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b128(rs, 16u * (uint32_t)(q * kSmThreads + tid), 0u, 0);
            Elem<T>::from_words((uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2], (uint32_t)w[3], v[q]);
        }
        const int head = a - lo, tail = hi - sl.body_end();
        edge = tid < head ? lo + tid : (tid - head < tail ? sl.body_end() + (tid - head) : -1);
        ve = edge >= 0 ? Elem<T>::load1(row + edge) : __builtin_nanf("");
#pragma unroll
        for (int q = 0; q < kVecs; ++q)
#pragma unroll
            for (int j = 0; j < VEC; ++j) {
                if (Tt != 1.0f) v[q][j] = v[q][j] / Tt;
                if (q * kSmThreads + tid >= nbody) v[q][j] = __builtin_nanf("");
            }
        if (Tt != 1.0f) ve = ve / Tt;
    }
};

// Part p of row r: the largest key and the sum of exp_det(y - that value) of its elements, left
// (3 words: key, sum low, sum high) at the start of EVERY part's slice of the row's
// probabilities, slot p of each.  softmax_write_kernel's workgroup for part q then reads the
// row's partial results from its own slice before it overwrites it, so the operation needs no
// workspace and no workgroup waits for another.
template <typename T>
__global__ __launch_bounds__(kSmThreads) void softmax_part_kernel(const T* logits, int64_t stride, int V,
                                                                  int part_len, int nparts,
                                                                  const float* temperature, float* probs) {
    constexpr int W = kSmThreads / kWave;
    __shared__ uint32_t redk[W];
    __shared__ double redd[W];
    const int r = blockIdx.x / nparts, p = blockIdx.x - r * nparts;
    const int tid = threadIdx.x, wave = tid >> 6;
    const float Tt = temperature ? temperature[r] : 1.0f;
    SoftmaxPart<T> sp;
    sp.load(logits + (size_t)r * stride, V, part_len, p, Tt);
    float mx = sp.ve;
#pragma unroll
    for (int q = 0; q < SoftmaxPart<T>::kVecs; ++q)
#pragma unroll
        for (int j = 0; j < SoftmaxPart<T>::VEC; ++j) mx = __builtin_fmaxf(mx, sp.v[q][j]);  // (NaN ignored)
    const uint32_t wk = wave_max_u32(key_of(mx));
    if ((tid & 63) == 0) redk[wave] = wk;
    __syncthreads();
    uint32_t mk = 0u;
#pragma unroll
    for (int w = 0; w < W; ++w) mk = mk > redk[w] ? mk : redk[w];
    const float m = mk ? val_of(mk) : -__builtin_inff();
    // exp_det is 0 for NaN: padding, NaN logits, and y - m of infinities
    double s = (double)exp_det(sp.ve - m);
#pragma unroll
    for (int q = 0; q < SoftmaxPart<T>::kVecs; ++q)
#pragma unroll
        for (int j = 0; j < SoftmaxPart<T>::VEC; ++j) s += (double)exp_det(sp.v[q][j] - m);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, kWave);
    if ((tid & 63) == 0) redd[wave] = s;
    __syncthreads();
    if (tid < nparts) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) t += redd[w];
        const uint64_t b = (uint64_t)__double_as_longlong(t);
        uint32_t* slot = reinterpret_cast<uint32_t*>(probs + (size_t)r * V + (size_t)tid * part_len) + 3 * p;
        slot[0] = mk;
        slot[1] = (uint32_t)b;
        slot[2] = (uint32_t)(b >> 32);
    }
}

template <typename T>
__global__ __launch_bounds__(kSmThreads) void softmax_write_kernel(const T* logits, int64_t stride, int V,
                                                                   int part_len, int nparts,
                                                                   const float* temperature, float* probs,
                                                                   float* row_max, float* log_sum) {
    constexpr int VEC = Elem<T>::kVec;
    const int r = blockIdx.x / nparts, p = blockIdx.x - r * nparts;
    const int tid = threadIdx.x, lane = tid & 63;
    const float Tt = temperature ? temperature[r] : 1.0f;
    float* out = probs + (size_t)r * V;
    // every wave combines the row's parts, one per lane (nparts <= 64)
    const uint32_t* slot = reinterpret_cast<const uint32_t*>(out + (size_t)p * part_len) + 3 * lane;
    const bool have = lane < nparts;
    const uint32_t pk = have ? slot[0] : 0u;
    const uint64_t pb = have ? ((uint64_t)slot[2] << 32) | slot[1] : 0ull;
    SoftmaxPart<T> sp;
    sp.load(logits + (size_t)r * stride, V, part_len, p, Tt);
    const uint32_t mk = wave_max_u32(pk);
    const float m = mk ? val_of(mk) : -__builtin_inff();  // (a row of NaN: the empty maximum)
    // a part without a finite maximum adds nothing, and without a finite row maximum S is 0
    const bool fin = __builtin_fabsf(m) < __builtin_inff() && pk > 0x007FFFFFu;
    double S = fin ? __longlong_as_double((long long)pb) * exp((double)val_of(pk) - (double)m) : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) S += __shfl_xor(S, o, kWave);
    const double inv = 1.0 / S;
    __syncthreads();  // every wave has read the slots: the slice may be written
    typedef float F4 __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int q = 0; q < SoftmaxPart<T>::kVecs; ++q) {
        const int vi = q * kSmThreads + tid;
        if (vi >= sp.nbody) break;
#pragma unroll
        for (int g = 0; g < VEC / 4; ++g) {
            F4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = (float)((double)exp_det(sp.v[q][4 * g + j] - m) * inv);
            *reinterpret_cast<F4*>(out + sp.a + vi * VEC + 4 * g) = o;
        }
    }
    if (sp.edge >= 0) out[sp.edge] = (float)((double)exp_det(sp.ve - m) * inv);
    if (p == 0 && tid == 0) {
        if (row_max) row_max[r] = m;
        if (log_sum) log_sum[r] = (float)log(S);
    }
}

// In-place vLLM-v1 penalties on fp32 rows: one workgroup per row, history deduplicated in a
// per-row hash in the workspace.
__global__ __launch_bounds__(kOpThreads) void penalties_kernel(KArgs a, float* logits) {
    const int r = blockIdx.x;
    const float rep = a.rep ? a.rep[r] : 1.0f;
    const float pres = a.pres ? a.pres[r] : 0.0f;
    const float freq = a.freq ? a.freq[r] : 0.0f;
    const float inv_rep = 1.0f / rep;
    const int np = a.prompt ? (a.plens ? min(max(a.plens[r], 0), a.pwidth) : a.pwidth) : 0;
    const int no = a.output ? (a.olens ? min(max(a.olens[r], 0), a.owidth) : a.owidth) : 0;
    const int hs = a.hs_row;
    if (hs == 0 || (np == 0 && no == 0)) return;
    uint32_t* hkey = a.hist_hash + (size_t)r * (size_t)hs * 4;
    uint32_t* hval = hkey + hs;
    for (int i = threadIdx.x; i < hs; i += kOpThreads) { hkey[i] = 0u; hval[i] = 0u; }
    __threadfence();
    __syncthreads();
    auto insert = [&](int t, uint32_t inc) {
        uint32_t s = ((uint32_t)t * 2654435761u) & (uint32_t)(hs - 1);
        for (int probe = 0; probe < hs; ++probe) {
            const uint32_t prev = atomicCAS(&hkey[s], 0u, (uint32_t)t + 1u);
            if (prev == 0u || prev == (uint32_t)t + 1u) {
                if (inc & 0x80000000u) atomicOr(&hval[s], 0x80000000u);
                else atomicAdd(&hval[s], inc);
                return;
            }
            s = (s + 1u) & (uint32_t)(hs - 1);
        }
    };
    for (int i = threadIdx.x; i < np; i += kOpThreads) {
        const int t = a.prompt[(size_t)r * a.pstride + i];
        if (t >= 0 && t < a.V) insert(t, 0x80000000u);
    }
    for (int i = threadIdx.x; i < no; i += kOpThreads) {
        const int t = a.output[(size_t)r * a.ostride + i];
        if (t >= 0 && t < a.V) insert(t, 1u);
    }
    __threadfence();
    __syncthreads();
    float* row = logits + (size_t)r * a.lstride;
    for (int s = threadIdx.x; s < hs; s += kOpThreads) {
        const uint32_t kk = __hip_atomic_load(&hkey[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!kk) continue;
        const uint32_t v = __hip_atomic_load(&hval[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int t = (int)kk - 1;
        row[t] = apply_penalty(row[t], (v >> 31) != 0u, v & 0x7FFFFFFFu, rep, inv_rep, freq, pres);
    }
    // The workspace is left as it was found (zeros).
    __syncthreads();
    for (int i = threadIdx.x; i < hs; i += kOpThreads) { hkey[i] = 0u; hval[i] = 0u; }
}

// Hash of f(x) over every fp32 x whose order key lies in [klo, khi]; same accumulation as the
// CPU oracle's checker (sum over inputs of bits(f(x)) * golden ^ bits(x)).
__global__ __launch_bounds__(256) void selftest_kernel(int fn, uint32_t klo, uint32_t khi,
                                                       unsigned long long* out) {
    __shared__ uint64_t red[4][2];
    uint64_t h = 0, c = 0;
    const uint64_t n = (uint64_t)khi - klo + 1ull;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256) {
        const uint32_t key = klo + (uint32_t)i;
        const uint32_t bits = (key & 0x80000000u) ? (key & 0x7FFFFFFFu) : ~key;
        const float x = u2f(bits);
        const float y = fn == 0 ? exp_det(x)
                      : (fn == 1 ? log_det(x) : (fn == 2 ? softcap_det(x, 1.0f, 1.0f) : round_f16(x)));
        h += ((uint64_t)f2u(y) * 0x9E3779B97F4A7C15ull) ^ (uint64_t)bits;
        c++;
    }
    h = wave_sum_u64(h);
    c = wave_sum_u64(c);
    if (lane_id() == 0) { red[threadIdx.x >> 6][0] = h; red[threadIdx.x >> 6][1] = c; }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t th = 0, tc = 0;
        for (int w = 0; w < 4; ++w) { th += red[w][0]; tc += red[w][1]; }
        atomicAdd(&out[0], (unsigned long long)th);
        atomicAdd(&out[1], (unsigned long long)tc);
    }
}

__global__ void fill_u32_kernel(uint32_t* p, size_t n, uint32_t v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// vws_token_state_update: one id per thread, counted (output) or flagged (prompt) in its row's
// word with a vector atomic (ids and rows may repeat within a call).
__global__ void token_state_kernel(uint32_t* st, int64_t stride, uint32_t* bits, int64_t bstride,
                                   int V, int n, const int32_t* rows, int row, const int32_t* tok,
                                   int kind) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    const int t = tok[i];
    const int rr = rows ? rows[i] : row;
    if (t < 0 || t >= V || rr < 0) return;
    uint32_t* w = st + (size_t)rr * (size_t)stride + (uint32_t)t;
    if (kind == VWS_STATE_OUTPUT) atomicAdd(w, 1u);
    else atomicOr(w, 0x80000000u);
    if (bits) atomicOr(bits + (size_t)rr * (size_t)bstride + ((uint32_t)t >> 5), 1u << (t & 31));
}

#define VWS_OPS_INST(T)                                                                             \
    template __global__ void argmax_kernel<T>(const T*, int64_t, int, int32_t*);                    \
    template __global__ void softmax_kernel<T>(const T*, int64_t, int, const float*, float*, float*, \
                                               float*);                                             \
    template __global__ void softmax_part_kernel<T>(const T*, int64_t, int, int, int, const float*,  \
                                                    float*);                                        \
    template __global__ void softmax_write_kernel<T>(const T*, int64_t, int, int, int, const float*, \
                                                     float*, float*, float*);
VWS_OPS_INST(float)
VWS_OPS_INST(uint16_t)
VWS_OPS_INST(_Float16)
#undef VWS_OPS_INST

}  // namespace vws
