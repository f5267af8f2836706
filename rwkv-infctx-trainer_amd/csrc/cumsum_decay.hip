// Cumulative-decay helper: from the raw decay parameter to the log-space
// tables of the chunked formulation (RWKV-v5/src/module/rwkv_inner.py:43-58,
// 72-79), in one fused pass.  log w = max(-exp(raw), ln 0.005) needs no log().
// One lane per (batch, chunk, channel); consecutive lanes are consecutive
// channels, so every row of every table is read and written coalesced.
#include "common.h"

namespace wkv {

__global__ __launch_bounds__(256) void cumsum_decay_kernel(int Bw, int Tlen, int C, int chunk, int per_token,
        const float *__restrict__ w, float *__restrict__ log_w, float *__restrict__ incl,
        float *__restrict__ inter, float *__restrict__ intra, float *__restrict__ chunk_sum)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    const int n = blockIdx.y, b = blockIdx.z, nchunk = Tlen / chunk;
    const size_t row0 = ((size_t)b * Tlen + (size_t)n * chunk) * C + c;
    const float fixed = per_token ? 0.f : log_decay(w[c], true);

    float total = 0.f;
    if (per_token) {
        for (int t = 0; t < chunk; t++) total += log_decay(w[row0 + (size_t)t * C], true);
    } else {
        for (int t = 0; t < chunk; t++) total += fixed;
    }
    if (chunk_sum) chunk_sum[((size_t)b * nchunk + n) * C + c] = total;

    float run = 0.f;
    for (int t = 0; t < chunk; t++) {
        const size_t o = row0 + (size_t)t * C;
        const float l = per_token ? log_decay(w[o], true) : fixed;
        run += l;
        if (log_w) log_w[o] = l;
        if (incl) incl[o] = run;
        if (inter) inter[o] = total - run;
        if (intra) intra[o] = run - l;
    }
}

// The same for the reference's chunk length (RWKV-v5/src/module/rwkv_inner.py:12), with or without the exponentiated
// tables.  Bound by the bytes written: 4 read and 16 written per element, 4 and 40 with every table in fp64.  Four
// wavefronts share a chunk, 32 tokens each, and a lane owns V neighbouring channels of them: w is read once (32
// independent loads per lane in flight), the running sum goes from one to the next through LDS, and every table is then written row by row
// in pieces of 64 V elements.  (One lane per channel walking all 128 tokens, w read twice, left ten wavefronts per
// compute unit: B2 T4096 C2560 with every fp64 table 304 us = 3.05 TB/s; now 200 us = 4.6 TB/s.)  V = 2 wherever the rows allow 8-byte accesses.
constexpr int DT_CHUNK = 128, DT_WAVES = 4, DT_TOK = DT_CHUNK / DT_WAVES;
template <class P, int V> __device__ __forceinline__ void store_table(P *p, const P (&x)[V]) {
    typedef P vec __attribute__((ext_vector_type(V)));
    vec v;
#pragma unroll
    for (int i = 0; i < V; i++) v[i] = x[i];
    __builtin_nontemporal_store(v, reinterpret_cast<vec *>(p));
}
template <class P> __device__ __forceinline__ void store_table(P *p, const P (&x)[1]) { __builtin_nontemporal_store(x[0], p); }

template <class P, bool FACTORS, int V>
__global__ __launch_bounds__(64 * DT_WAVES) void decay_tables_128(int Tlen, int C, int per_token,
        const float *__restrict__ w, float *__restrict__ log_w, float *__restrict__ incl, float *__restrict__ inter,
        float *__restrict__ intra, float *__restrict__ chunk_sum, float *__restrict__ ws_exp, float *__restrict__ inter_exp,
        float *__restrict__ intra_exp, P *__restrict__ r_decay, P *__restrict__ k_inv_decay)
{
    __shared__ float part[DT_WAVES][64 * V];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int c = (blockIdx.x * 64 + lane) * V;              // (C is a multiple of V)
    const int n = blockIdx.y, b = blockIdx.z, nchunk = Tlen / DT_CHUNK;
    const bool in = c < C;
    const size_t row0 = ((size_t)b * Tlen + (size_t)n * DT_CHUNK + wv * DT_TOK) * C + (in ? c : 0);
    float l[DT_TOK][V];
    if (per_token) {
#pragma unroll
        for (int t = 0; t < DT_TOK; t++) {
            if constexpr (V == 2) {
                const float2 x = *reinterpret_cast<const float2 *>(w + row0 + (size_t)t * C);
                l[t][0] = x.x; l[t][1] = x.y;
            } else {
                l[t][0] = w[row0 + (size_t)t * C];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < V; i++) {
        const float fixed = per_token ? 0.f : log_decay(w[(in ? c : 0) + i], true);
#pragma unroll
        for (int t = 0; t < DT_TOK; t++) l[t][i] = per_token ? log_decay(l[t][i], true) : fixed;
    }
    // The running sum goes through the wavefronts in turn, each adding its tokens to where the one before it ended: one sum from
    // the chunk's first token to its last, so that the total is exactly the last token's running sum (inter there exactly
    // 0) and no running sum rises.  The three waits are hidden by the other workgroups.
    float run[V], total[V], mid[V];
#pragma unroll
    for (int i = 0; i < V; i++) run[i] = 0.f;
#pragma unroll
    for (int q = 0; q < DT_WAVES; q++) {
        if (q == wv) {
            if (q > 0)
#pragma unroll
                for (int i = 0; i < V; i++) run[i] = part[q - 1][lane * V + i];
#pragma unroll
            for (int i = 0; i < V; i++) {
                float s = run[i];
#pragma unroll
                for (int t = 0; t < DT_TOK; t++) s += l[t][i];
                part[q][lane * V + i] = s;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < V; i++) {
        mid[i] = part[DT_WAVES / 2 - 1][lane * V + i];          // exclusive running sum at token 64
        total[i] = part[DT_WAVES - 1][lane * V + i];
    }
    if (!in) return;
    if (wv == 0) {
        const size_t o = ((size_t)b * nchunk + n) * C + c;
#pragma unroll
        for (int i = 0; i < V; i++) {
            if (chunk_sum) chunk_sum[o + i] = total[i];
            if (FACTORS && ws_exp) ws_exp[o + i] = expf(total[i]);
        }
    }
#pragma unroll 4
    for (int t = 0; t < DT_TOK; t++) {
        const size_t o = row0 + (size_t)t * C;
        float f_inter[V], f_intra[V], e_inter[V], e_intra[V], lw[V];
        P rd[V], ki[V];
#pragma unroll
        for (int i = 0; i < V; i++) {
            const float excl = run[i];
            lw[i] = l[t][i];
            run[i] += lw[i];
            f_inter[i] = total[i] - run[i];
            f_intra[i] = run[i] - lw[i];                     // as the reference forms it (:79), not the shifted sum
            if (FACTORS) {
                e_inter[i] = expf(f_inter[i]);
                e_intra[i] = expf(f_intra[i]);
                rd[i] = exp((P)(excl - mid[i]));
                ki[i] = exp((P)(mid[i] - run[i]));
            }
        }
        if (log_w) store_table(log_w + o, lw);
        if (incl) store_table(incl + o, run);
        if (inter) store_table(inter + o, f_inter);
        if (intra) store_table(intra + o, f_intra);
        if (FACTORS) {
            if (inter_exp) store_table(inter_exp + o, e_inter);
            if (intra_exp) store_table(intra_exp + o, e_intra);
            if (r_decay) store_table(r_decay + o, rd);
            if (k_inv_decay) store_table(k_inv_decay + o, ki);
        }
    }
}

// All outputs of the helper, including the exponentiated tables (rwkv_inner.py:80-82) and the two factors of the
// intra-chunk product re-centred on the chunk's middle token (:91-93), which the reference forms in fp64
// (precision = 64: their exponents reach +-64 * 5.3) or fp32 (precision = 32, for chunk lengths up to 32).
template <class P>
__global__ __launch_bounds__(256) void cumsum_decay_factors(int Bw, int Tlen, int C, int chunk, int per_token,
        const float *__restrict__ w, float *__restrict__ log_w, float *__restrict__ incl, float *__restrict__ inter,
        float *__restrict__ intra, float *__restrict__ chunk_sum, float *__restrict__ ws_exp, float *__restrict__ inter_exp,
        float *__restrict__ intra_exp, P *__restrict__ r_decay, P *__restrict__ k_inv_decay)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    const int n = blockIdx.y, b = blockIdx.z, nchunk = Tlen / chunk;
    const size_t row0 = ((size_t)b * Tlen + (size_t)n * chunk) * C + c;
    const float fixed = per_token ? 0.f : log_decay(w[c], true);
    float total = 0.f, mid = 0.f;              // mid = exclusive running sum at token chunk/2
    for (int t = 0; t < chunk; t++) {
        if (t == chunk / 2) mid = total;
        total += per_token ? log_decay(w[row0 + (size_t)t * C], true) : fixed;
    }
    if (chunk_sum) chunk_sum[((size_t)b * nchunk + n) * C + c] = total;
    if (ws_exp) ws_exp[((size_t)b * nchunk + n) * C + c] = expf(total);
    float run = 0.f;
    for (int t = 0; t < chunk; t++) {
        const size_t o = row0 + (size_t)t * C;
        const float l = per_token ? log_decay(w[o], true) : fixed;
        const float excl = run;
        run += l;
        if (log_w) log_w[o] = l;
        if (incl) incl[o] = run;
        if (inter) inter[o] = total - run;
        if (intra) intra[o] = run - l;                       // as the reference forms it (:79), not the shifted sum
        if (inter_exp) inter_exp[o] = expf(total - run);
        if (intra_exp) intra_exp[o] = expf(run - l);
        if (r_decay) r_decay[o] = exp((P)(excl - mid));
        if (k_inv_decay) k_inv_decay[o] = exp((P)(mid - run));
    }
}

// 8-byte (fp64: 16-byte) accesses to pairs of channels: every row of every table then starts on their boundary
static bool pairs_aligned(int C, std::initializer_list<const void *> tables4, std::initializer_list<const void *> tables8 = {}) {
    uintptr_t a = C & 1;
    for (const void *p : tables4) a |= reinterpret_cast<uintptr_t>(p) & 7u;
    for (const void *p : tables8) a |= reinterpret_cast<uintptr_t>(p) & 15u;
    return a == 0;
}
template <class P, bool FACTORS>
static void decay_tables_128_launch(hipStream_t s, bool pairs, int Bw, int Tlen, int C, int per_token, const float *w, float *log_w,
                                    float *incl, float *inter, float *intra, float *chunk_sum, float *ws_exp = nullptr,
                                    float *inter_exp = nullptr, float *intra_exp = nullptr, void *r_decay = nullptr,
                                    void *k_inv_decay = nullptr) {
    const int V = pairs ? 2 : 1;
    const dim3 grid((C + 64 * V - 1) / (64 * V), Tlen / DT_CHUNK, Bw), block(64 * DT_WAVES);
#define WKV_TABLES(V_)                                                                                                      \
    hipLaunchKernelGGL((decay_tables_128<P, FACTORS, V_>), grid, block, 0, s, Tlen, C, per_token, w, log_w, incl, inter, intra, \
                       chunk_sum, ws_exp, inter_exp, intra_exp, (P *)r_decay, (P *)k_inv_decay)
    if (pairs) WKV_TABLES(2); else WKV_TABLES(1);
#undef WKV_TABLES
}

hipError_t cumsum_decay_factors_launch(hipStream_t s, int Bw, int Tlen, int C, int chunk, int per_token, int precision,
                                       const float *w, float *log_w, float *incl, float *inter, float *intra, float *chunk_sum,
                                       float *ws_exp, float *inter_exp, float *intra_exp, void *r_decay, void *k_inv_decay) {
    dim3 grid((C + 255) / 256, Tlen / chunk, Bw);
    if (chunk == DT_CHUNK) {
        const bool wide = precision == 64;
        const bool pairs = pairs_aligned(C, {w, log_w, incl, inter, intra, inter_exp, intra_exp, wide ? nullptr : r_decay, wide ? nullptr : k_inv_decay},
                                         {wide ? r_decay : nullptr, wide ? k_inv_decay : nullptr});
        if (wide)
            decay_tables_128_launch<double, true>(s, pairs, Bw, Tlen, C, per_token, w, log_w, incl, inter, intra, chunk_sum, ws_exp,
                                                  inter_exp, intra_exp, r_decay, k_inv_decay);
        else
            decay_tables_128_launch<float, true>(s, pairs, Bw, Tlen, C, per_token, w, log_w, incl, inter, intra, chunk_sum, ws_exp,
                                                 inter_exp, intra_exp, r_decay, k_inv_decay);
        return hipGetLastError();
    }
    if (precision == 64)
        hipLaunchKernelGGL(cumsum_decay_factors<double>, grid, dim3(256), 0, s, Bw, Tlen, C, chunk, per_token, w, log_w, incl,
                           inter, intra, chunk_sum, ws_exp, inter_exp, intra_exp, (double *)r_decay, (double *)k_inv_decay);
    else
        hipLaunchKernelGGL(cumsum_decay_factors<float>, grid, dim3(256), 0, s, Bw, Tlen, C, chunk, per_token, w, log_w, incl,
                           inter, intra, chunk_sum, ws_exp, inter_exp, intra_exp, (float *)r_decay, (float *)k_inv_decay);
    return hipGetLastError();
}

hipError_t cumsum_decay_launch(hipStream_t s, int Bw, int Tlen, int C, int chunk, int per_token, const float *w,
                               float *log_w, float *incl, float *inter, float *intra, float *chunk_sum) {
    dim3 grid((C + 255) / 256, Tlen / chunk, Bw);
    if (chunk == DT_CHUNK) {
        decay_tables_128_launch<float, false>(s, pairs_aligned(C, {w, log_w, incl, inter, intra}), Bw, Tlen, C, per_token, w, log_w,
                                              incl, inter, intra, chunk_sum);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(cumsum_decay_kernel, grid, dim3(256), 0, s, Bw, Tlen, C, chunk, per_token, w, log_w, incl, inter,
                       intra, chunk_sum);
    return hipGetLastError();
}

}  // namespace wkv
