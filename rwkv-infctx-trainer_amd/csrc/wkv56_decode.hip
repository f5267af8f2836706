// One token of WKV5 / WKV6 for every (batch, head): the serving loop's call.
//
//     y[j] = sum_i r[i] (S[i][j] + u[i] k[i] v[j]),    S[i][j] <- w[i] S[i][j] + k[i] v[j]
//
// (RWKV-v5/src/module/rwkv_inner.py:28-32.)  Bound by the state, 16 KiB in and 16 KiB out per head: one workgroup per
// head, lane (key group, four value columns), so that a wavefront's four 16-byte loads are whole kilobytes and all of a
// head's state is in flight at once; nothing of a token is staged in LDS except the four wavefronts' sums.  The token
// loop's kernel (rec_forward) staged 16 tokens for the one it had: B64 H32 13.0 us; here 10.6 us = 6.4 TB/s.  The raw decay is read in
// the type it has, fp32 or that of r, k and v.
#include "common.h"

namespace wkv {

template <class T, class W, bool PER_TOKEN_W>
__global__ __launch_bounds__(256) void decode56(int H, const T *__restrict__ r, const T *__restrict__ k, const T *__restrict__ v,
        const W *__restrict__ wraw, const float *__restrict__ u, const float *s_in, T *__restrict__ y, float *s_out, int floor_decay)
{
    __shared__ __align__(16) float part[4][HEAD];
    const int bh = blockIdx.x, h = bh % H, tid = threadIdx.x, kq = tid >> 4, c4 = 4 * (tid & 15);
    const size_t base = (size_t)bh * HEAD, so = (size_t)bh * HEAD * HEAD;
    // (s_out may be s_in: a lane writes the elements it has read)
    float4 S[4];
#pragma unroll
    for (int i = 0; i < 4; i++) S[i] = *reinterpret_cast<const float4 *>(s_in + so + (kq + 16 * i) * HEAD + c4);
    float v4[4], acc[4] = {0.f, 0.f, 0.f, 0.f}, bonus = 0.f;
    load4(v + base + c4, v4);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int key = kq + 16 * i;
        const float ri = to_float(r[base + key]), ki = to_float(k[base + key]);
        const float wi = __expf(log_decay(to_float(wraw[(PER_TOKEN_W ? base : (size_t)h * HEAD) + key]), floor_decay));
        bonus = fmaf(ri * u[h * HEAD + key], ki, bonus);
        float s[4] = {S[i].x, S[i].y, S[i].z, S[i].w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            acc[e] = fmaf(ri, s[e], acc[e]);
            s[e] = fmaf(wi, s[e], ki * v4[e]);
        }
        *reinterpret_cast<float4 *>(s_out + so + key * HEAD + c4) = make_float4(s[0], s[1], s[2], s[3]);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        acc[e] = fmaf(v4[e], bonus, acc[e]);
        acc[e] += __shfl_xor(acc[e], 16);
        acc[e] += __shfl_xor(acc[e], 32);
    }
    if ((tid & 63) < 16) *reinterpret_cast<float4 *>(&part[tid >> 6][c4]) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    __syncthreads();
    if (tid < HEAD) y[base + tid] = from_float<T>((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]));
}

// w_dtype: that of the raw decay (wkv_dtype), fp32 or the same as `dtype`
static hipError_t decode_launch(hipStream_t s, int dtype, int w_dtype, bool per_token, int BH, int H, const void *r, const void *k,
                                const void *v, const void *w, const float *u, const float *s_in, void *y, float *s_out, int floor_decay) {
    prof_begin(KID_REC_FORWARD, s);
#define WKV_DECODE(T, W, PT)                                                                                                  \
    hipLaunchKernelGGL((decode56<T, W, PT>), dim3(BH), dim3(256), 0, s, H, (const T *)r, (const T *)k, (const T *)v, (const W *)w, \
                       u, s_in, (T *)y, s_out, floor_decay)
#define WKV_DECODE_T(T)                                      \
    do {                                                     \
        if (!per_token) WKV_DECODE(T, float, false);         \
        else if (w_dtype == 0) WKV_DECODE(T, float, true);   \
        else WKV_DECODE(T, T, true);                         \
    } while (0)
    if (dtype == 0) WKV_DECODE_T(float);
    else if (dtype == 1) WKV_DECODE_T(bf16);
    else WKV_DECODE_T(f16);
#undef WKV_DECODE_T
#undef WKV_DECODE
    prof_end(KID_REC_FORWARD, s);
    return hipGetLastError();
}

}  // namespace wkv
