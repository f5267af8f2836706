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
// wavefronts share 64 channels of a chunk, 32 tokens each: w is read once (32 independent loads per lane in flight), the running
// sum goes from one to the next through LDS, and every table is then written row by row.  One lane per channel walking all
// 128 tokens left ten wavefronts per compute unit: B2 T4096 C2560 with every fp64 table 293 us, log tables 85 us; now 163 and 64 us
// (5.6 and 6.6 TB/s).  The tokens' loops are unrolled whole: left at four tokens the log decays, indexed by a variable, sit in
// scratch memory (two channels a lane: 182 and 98 us).
// COLS groups of four wavefronts side by side make a workgroup, so that its pieces of the rows are 256 COLS bytes long.
constexpr int DT_CHUNK = 128, DT_WAVES = 4, DT_TOK = DT_CHUNK / DT_WAVES;
// LINES: the rows start on cache lines.  Past the caches then (B4 T4096 C2560 log tables 124 us against 172); where a line
// holds the end of one workgroup's piece and the start of the next one's it has to wait for both in a cache (C 2049: 474 against 593).
template <bool LINES, class P> __device__ __forceinline__ void store_table(P *p, P x) {
    if (LINES) __builtin_nontemporal_store(x, p);
    else *p = x;
}

template <class P, bool FACTORS, int COLS, bool LINES>
__global__ __launch_bounds__(64 * DT_WAVES * COLS) void decay_tables_128(int Tlen, int C, int per_token,
        const float *__restrict__ w, float *__restrict__ log_w, float *__restrict__ incl, float *__restrict__ inter,
        float *__restrict__ intra, float *__restrict__ chunk_sum, float *__restrict__ ws_exp, float *__restrict__ inter_exp,
        float *__restrict__ intra_exp, P *__restrict__ r_decay, P *__restrict__ k_inv_decay)
{
    __shared__ float part[DT_WAVES][64 * COLS];
    const int lane = threadIdx.x % (64 * COLS), wv = threadIdx.x / (64 * COLS);
    const int c = blockIdx.x * 64 * COLS + lane;
    const int n = blockIdx.y, b = blockIdx.z, nchunk = Tlen / DT_CHUNK;
    const bool in = c < C;
    const size_t row0 = ((size_t)b * Tlen + (size_t)n * DT_CHUNK + wv * DT_TOK) * C + (in ? c : 0);
    float l[DT_TOK];
    if (per_token) {
#pragma unroll
        for (int t = 0; t < DT_TOK; t++) l[t] = w[row0 + (size_t)t * C];
    }
    const float fixed = per_token ? 0.f : log_decay(w[in ? c : 0], true);
#pragma unroll
    for (int t = 0; t < DT_TOK; t++) l[t] = per_token ? log_decay(l[t], true) : fixed;
    // The running sum goes through the wavefronts in turn, each adding its tokens to where the one before it ended: one sum from
    // the chunk's first token to its last, so that the total is exactly the last token's running sum (inter there exactly
    // 0) and no running sum rises.  The three waits are hidden by the other workgroups.
    float run = 0.f;
#pragma unroll
    for (int q = 0; q < DT_WAVES; q++) {
        if (q == wv) {
            if (q > 0) run = part[q - 1][lane];
            float s = run;
#pragma unroll
            for (int t = 0; t < DT_TOK; t++) s += l[t];
            part[q][lane] = s;
        }
        __syncthreads();
    }
    const float mid = part[DT_WAVES / 2 - 1][lane];          // exclusive running sum at token 64
    const float total = part[DT_WAVES - 1][lane];
    if (!in) return;
    if (wv == 0) {
        const size_t o = ((size_t)b * nchunk + n) * C + c;
        if (chunk_sum) chunk_sum[o] = total;
        if (FACTORS && ws_exp) ws_exp[o] = expf(total);
    }
#pragma unroll
    for (int t = 0; t < DT_TOK; t++) {
        const size_t o = row0 + (size_t)t * C;
        const float excl = run, lw = l[t];
        run += lw;
        const float f_inter = total - run, f_intra = run - lw;          // as the reference forms it (:79), not the shifted sum
        if (log_w) store_table<LINES>(log_w + o, lw);
        if (incl) store_table<LINES>(incl + o, run);
        if (inter) store_table<LINES>(inter + o, f_inter);
        if (intra) store_table<LINES>(intra + o, f_intra);
        if (FACTORS) {
            if (inter_exp) store_table<LINES>(inter_exp + o, expf(f_inter));
            if (intra_exp) store_table<LINES>(intra_exp + o, expf(f_intra));
            if (r_decay) store_table<LINES>(r_decay + o, exp((P)(excl - mid)));
            if (k_inv_decay) store_table<LINES>(k_inv_decay + o, exp((P)(mid - run)));
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

// Four columns of wavefronts per workgroup where the rows do not start on cache lines (fewer lines are then shared between
// workgroups: B8 T4096 C2049 log tables 358 us, with one column 474; C801, two chunks of rows, 13.1 and 9.6: only from two workgroups per
// compute unit on); two where they do and there are many (B8 T4096 C2560 322 against 332, B4 125 against 124, C512 8.5 against 8.5).
template <class P, bool FACTORS>
static void decay_tables_128_launch(hipStream_t s, int Bw, int Tlen, int C, int per_token, const float *w, float *log_w,
                                    float *incl, float *inter, float *intra, float *chunk_sum, float *ws_exp = nullptr,
                                    float *inter_exp = nullptr, float *intra_exp = nullptr, void *r_decay = nullptr,
                                    void *k_inv_decay = nullptr) {
    const bool lines = C % 32 == 0;
    const long four = (long)Bw * (Tlen / DT_CHUNK) * ((C + 255) / 256), ncu = cu_count();
#define WKV_TABLES(COLS_, LINES_)                                                                                           \
    hipLaunchKernelGGL((decay_tables_128<P, FACTORS, COLS_, LINES_>), dim3((C + 64 * COLS_ - 1) / (64 * COLS_), Tlen / DT_CHUNK, Bw), \
                       dim3(64 * DT_WAVES * COLS_), 0, s, Tlen, C, per_token, w, log_w, incl, inter, intra, chunk_sum, ws_exp, inter_exp, \
                       intra_exp, (P *)r_decay, (P *)k_inv_decay)
    if (lines && four >= 8 * ncu) WKV_TABLES(2, true);
    else if (lines) WKV_TABLES(1, true);
    else if (four >= 2 * ncu) WKV_TABLES(4, false);
    else WKV_TABLES(1, false);
#undef WKV_TABLES
}

hipError_t cumsum_decay_factors_launch(hipStream_t s, int Bw, int Tlen, int C, int chunk, int per_token, int precision,
                                       const float *w, float *log_w, float *incl, float *inter, float *intra, float *chunk_sum,
                                       float *ws_exp, float *inter_exp, float *intra_exp, void *r_decay, void *k_inv_decay) {
    dim3 grid((C + 255) / 256, Tlen / chunk, Bw);
    if (chunk == DT_CHUNK) {
        if (precision == 64)
            decay_tables_128_launch<double, true>(s, Bw, Tlen, C, per_token, w, log_w, incl, inter, intra, chunk_sum, ws_exp,
                                                  inter_exp, intra_exp, r_decay, k_inv_decay);
        else
            decay_tables_128_launch<float, true>(s, Bw, Tlen, C, per_token, w, log_w, incl, inter, intra, chunk_sum, ws_exp,
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
        decay_tables_128_launch<float, false>(s, Bw, Tlen, C, per_token, w, log_w, incl, inter, intra, chunk_sum);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(cumsum_decay_kernel, grid, dim3(256), 0, s, Bw, Tlen, C, chunk, per_token, w, log_w, incl, inter,
                       intra, chunk_sum);
    return hipGetLastError();
}

}  // namespace wkv
