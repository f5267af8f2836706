// The layer of a serving loop: one token per sequence, a few rows (sequences) at a time, bf16.  What a row costs is the
// weights, read once; as library products, element-wise passes and dtype conversions a v6 layer of one row was some 45
// launches (H32: 526 us, of which the weights need 22 us).  Here it is seven kernels:
//
//   rows_products   any number of products  out = f(x' W)  of up to 64 rows with weights of their own, in one launch;
//                   x' may be the token-shift mix of x, formed where it is read (RWKV-v5/src/module/TimeMix.py:295-298,
//                   ChannelMix.py:46-47), and f one of the activations that follow a projection in a layer
//   lora_mix_rows   the five data-dependent mixes of the v6 TimeMix (RWKV-v6/src/module/TimeMix.py:264-276)
//   timemix_head    per head: the v6 decay's second LoRA product, the operator's single step, ln_x and the gate
//                   (RWKV-v6/src/module/TimeMix.py:280-298, RWKV-v5/src/module/TimeMix.py:309-320)
//
// Everything between two tensors of memory is fp32.
#include "common.h"

namespace wkv {
namespace rows {

typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int MAX_ROWS = 64, MAX_JOBS = 8;
struct Job {
    const bf16 *w;          // k_major ? [K][N] : [N][K]
    const bf16 *x;          // [rows][K]
    const bf16 *shift;      // [rows][K], with mix
    const bf16 *mix;        // [K], or NULL: x as it is
    const bf16 *mul;        // [rows][N], ACT_SIGMOID_MUL
    bf16 *out;              // [rows][N]
    int n, k_major, lerp, act;
};
struct Jobs { Job j[MAX_JOBS]; int count; };
enum { ACT_NONE = 0, ACT_TANH = 1, ACT_RELU_SQUARE = 2, ACT_SIGMOID_MUL = 3 };

__device__ __forceinline__ f4 mma(s8 a, s8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}
__device__ __forceinline__ float bf(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ float sigmoid(float x) { return __builtin_amdgcn_rcpf(1.f + exp2_fast(-LOG2E * x)); }
__device__ __forceinline__ float round_bf16(float x) { return bf(bf16_bits(x)); }

// Eight values of the mixed row: x + (shift - x) d, rounded to bf16 as the mixing pass leaves it
__device__ __forceinline__ s8 mixed(s8 x, s8 xx, s8 c, int lerp) {
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const float a = bf((uint16_t)x[e]), d = lerp ? 1.f - bf((uint16_t)c[e]) : bf((uint16_t)c[e]);
        o[e] = fmaf(bf((uint16_t)xx[e]) - a, d, a);
    }
    const uint4 p = make_uint4(bf16_pack2(o[0], o[1]), bf16_pack2(o[2], o[3]), bf16_pack2(o[4], o[5]), bf16_pack2(o[6], o[7]));
    return __builtin_bit_cast(s8, p);
}

// One wavefront's share of a 16-column tile: the 64-deep chunks wv, wv + WAVES, ... of the contraction.  The weights
// are the A operand (their columns are the MFMA's rows), the rows of x the B operand: lane (kg = lane/16, n = lane%16)
// supplies weight row n and x row n, eight consecutive k each.
template <int MT, int WAVES, int U, bool MIX, bool K_MAJOR>
__device__ __forceinline__ void accumulate(const Job &job, int tile, int rows, int K, int wv, int kg, int n, f4 (&acc)[MT]) {
    const int chunks = K / 64;
    const bf16 *w = job.w + (K_MAJOR ? (size_t)16 * tile + n + (size_t)(8 * kg) * job.n : (size_t)(16 * tile + n) * K + 8 * kg);
    size_t xo[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) xo[mt] = (size_t)min(16 * mt + n, rows - 1) * K + 8 * kg;
    for (int c0 = wv; c0 < chunks; c0 += U * WAVES) {
        s8 a[U][2], b[U][2][MT], bs[MIX ? U : 1][2][MT], bc[MIX ? U : 1][2];
#pragma unroll
        for (int i = 0; i < U; i++) {
            const int c = min(c0 + i * WAVES, chunks - 1);           // (a chunk past the end is read again and not used)
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                const int k = 64 * c + 32 * hf;
                if (K_MAJOR) {
#pragma unroll
                    for (int e = 0; e < 8; e++) a[i][hf][e] = (short)w[(size_t)(k + e) * job.n].bits;
                } else {
                    a[i][hf] = *reinterpret_cast<const s8 *>(w + k);
                }
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    b[i][hf][mt] = *reinterpret_cast<const s8 *>(job.x + xo[mt] + k);
                    if (MIX) bs[i][hf][mt] = *reinterpret_cast<const s8 *>(job.shift + xo[mt] + k);
                }
                if (MIX) bc[i][hf] = *reinterpret_cast<const s8 *>(job.mix + 8 * kg + k);
            }
        }
#pragma unroll
        for (int i = 0; i < U; i++)
            if (c0 + i * WAVES < chunks) {
#pragma unroll
                for (int hf = 0; hf < 2; hf++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        acc[mt] = mma(a[i][hf], MIX ? mixed(b[i][hf][mt], bs[i][hf][mt], bc[i][hf], job.lerp) : b[i][hf][mt], acc[mt]);
            }
    }
}

// A workgroup per 16 columns; its wavefronts share the contraction and meet in LDS.  Bound by the weights: every
// wavefront keeps up to 8 KB of them in flight, and the chunks of a row are dealt out so that the wavefronts of a
// workgroup read 64 WAVES consecutive elements of it together.  (x, up to 64 rows, comes out of the caches.)
template <int MT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void rows_products(int rows, int K, Jobs jobs) {
    __shared__ __align__(16) f4 part[WAVES][MT][64];
    int tile = blockIdx.x, ji = 0;
    while (tile >= jobs.j[ji].n / 16) tile -= jobs.j[ji++].n / 16;     // (the grid is the sum of all tiles)
    const Job job = jobs.j[ji];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, n = lane & 15;
    f4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[mt] = f4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = MT == 1 ? 4 : 2, UM = MT == 1 ? 2 : 1;
    if (job.k_major) {
        if (job.mix) accumulate<MT, WAVES, UM, true, true>(job, tile, rows, K, wv, kg, n, acc);
        else accumulate<MT, WAVES, UM, false, true>(job, tile, rows, K, wv, kg, n, acc);
    } else {
        if (job.mix) accumulate<MT, WAVES, UM, true, false>(job, tile, rows, K, wv, kg, n, acc);
        else accumulate<MT, WAVES, U, false, false>(job, tile, rows, K, wv, kg, n, acc);
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) part[wv][mt][lane] = acc[mt];
    __syncthreads();
    if (wv >= MT) return;
    f4 s = part[0][wv][lane];
#pragma unroll
    for (int i = 1; i < WAVES; i++) s += part[i][wv][lane];
    const int m = 16 * wv + n;                          // the lane holds columns 16 tile + 4 kg .. +3 of row m
    if (m >= rows) return;
    const size_t o = (size_t)m * job.n + 16 * tile + 4 * kg;
    float y[4] = {s[0], s[1], s[2], s[3]};
    if (job.act == ACT_TANH) {
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = tanhf(y[e]);
    } else if (job.act == ACT_RELU_SQUARE) {
#pragma unroll
        for (int e = 0; e < 4; e++) { const float p = fmaxf(round_bf16(y[e]), 0.f); y[e] = p * p; }
    } else if (job.act == ACT_SIGMOID_MUL) {
        float q[4];
        load4(job.mul + o, q);
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = sigmoid(q[e]) * round_bf16(y[e]);
    }
    store4(job.out + o, y);
}

// out[j] = x + (shift - x) (maa_j + act_j w2_j): a wavefront per mix and 16 channels, whose 32-deep product is one MFMA
// per 16 rows.  act [rows][5][32]; w2 [5][32][C].
struct Maa { const bf16 *p[5]; };
__global__ __launch_bounds__(320) void lora_mix_rows(int rows, int C, const bf16 *__restrict__ x, const bf16 *__restrict__ shift,
        Maa maa, const bf16 *__restrict__ act, const bf16 *__restrict__ w2, bf16 *__restrict__ out)
{
    const int lane = threadIdx.x & 63, j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, n = lane & 15;
    const int c0 = 16 * blockIdx.x;
    s8 a;
    const bf16 *w = w2 + ((size_t)j * 32 + 8 * kg) * C + c0 + n;
#pragma unroll
    for (int e = 0; e < 8; e++) a[e] = (short)w[(size_t)e * C].bits;
    float d[4];
    load4(maa.p[j] + c0 + 4 * kg, d);
    for (int m0 = 0; m0 < rows; m0 += 16) {
        const int m = m0 + n, mc = min(m, rows - 1);
        const s8 b = *reinterpret_cast<const s8 *>(act + ((size_t)mc * 5 + j) * 32 + 8 * kg);
        const size_t o = (size_t)mc * C + c0 + 4 * kg;
        float xv[4], xx[4], y[4];
        load4(x + o, xv);
        load4(shift + o, xx);
        const f4 dyn = mma(a, b, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = fmaf(xx[e] - xv[e], d[e] + dyn[e], xv[e]);
        if (m < rows) store4(out + (size_t)j * rows * C + o, y);
    }
}

// One workgroup per (row, head), lane (key group, four value columns) as in decode56.  lora != NULL (v6): the raw decay
// of the head's channels is time_decay + lora[row] w2 (64 deep); NULL (v5): time_decay itself.
__global__ __launch_bounds__(256) void timemix_head(int H, const bf16 *__restrict__ r, const bf16 *__restrict__ k, const bf16 *__restrict__ v,
        const bf16 *__restrict__ gate, const bf16 *__restrict__ time_decay, const bf16 *__restrict__ lora, const bf16 *__restrict__ w2,
        const bf16 *__restrict__ u, const bf16 *__restrict__ ln_w, const bf16 *__restrict__ ln_b, float scale, float eps,
        const float *s_in, float *s_out, bf16 *__restrict__ out)
{
    __shared__ __align__(16) float part[4][HEAD], dec[HEAD];
    const int row = blockIdx.x / H, h = blockIdx.x % H, C = H * HEAD, tid = threadIdx.x, kq = tid >> 4, c4 = 4 * (tid & 15);
    const size_t base = (size_t)row * C + h * HEAD, so = (size_t)blockIdx.x * HEAD * HEAD;
    float4 S[4];
#pragma unroll
    for (int i = 0; i < 4; i++) S[i] = *reinterpret_cast<const float4 *>(s_in + so + (kq + 16 * i) * HEAD + c4);
    {
        const int ch = tid & 63, q = tid >> 6;
        float a = 0.f;
        if (lora) {
#pragma unroll
            for (int e = 0; e < 16; e++)
                a = fmaf(to_float(lora[(size_t)row * 64 + 16 * q + e]), to_float(w2[(size_t)(16 * q + e) * C + h * HEAD + ch]), a);
        }
        part[q][ch] = a;
        __syncthreads();
        if (tid < HEAD)
            dec[tid] = __expf(log_decay(to_float(time_decay[h * HEAD + tid]) + ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid])), false));
        __syncthreads();
    }
    float v4[4], acc[4] = {0.f, 0.f, 0.f, 0.f}, bonus = 0.f;
    load4(v + base + c4, v4);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int key = kq + 16 * i;
        const float ri = to_float(r[base + key]), ki = to_float(k[base + key]), wi = dec[key];
        bonus = fmaf(ri * to_float(u[h * HEAD + key]), ki, bonus);
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
    if (tid >= HEAD) return;
    const float y = scale * ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]));
    float s = y;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
    const float dy = y - s * (1.f / HEAD);
    float q = dy * dy;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) q += __shfl_xor(q, o);
    const int c = h * HEAD + tid;
    const float g = to_float(gate[base + tid]);
    const float z = fmaf(dy * rsqrtf(q * (1.f / HEAD) + eps), to_float(ln_w[c]), to_float(ln_b[c]));
    out[base + tid] = from_float<bf16>(z * g * sigmoid(g));
}

// Sixteen wavefronts per tile where the tiles do not fill the compute units, eight otherwise: the wavefronts' number is
// what keeps memory requests in flight, and meeting in LDS costs more the more of them meet.
static hipError_t rows_products_launch(hipStream_t s, int rows, int K, const Jobs &jobs) {
    int tiles = 0;
    for (int i = 0; i < jobs.count; i++) tiles += jobs.j[i].n / 16;
    const bool wide = tiles < 2 * cu_count();
#define WKV_ROWS(MT)                                                                                                  \
    do {                                                                                                              \
        if (wide) hipLaunchKernelGGL((rows_products<MT, 16>), dim3(tiles), dim3(1024), 0, s, rows, K, jobs);          \
        else hipLaunchKernelGGL((rows_products<MT, 8>), dim3(tiles), dim3(512), 0, s, rows, K, jobs);                 \
    } while (0)
    if (rows <= 16) WKV_ROWS(1);
    else if (rows <= 32) WKV_ROWS(2);
    else WKV_ROWS(4);
#undef WKV_ROWS
    return hipGetLastError();
}

}  // namespace rows
}  // namespace wkv
