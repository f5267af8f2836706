// The contractions over the channels that the v6 TimeMix's two LoRAs have:  out = f(x w)  with x (rows, C) and 160, 64 or
// five times 32 columns (RWKV-v6/src/module/TimeMix.py:264,280-281 and their backward), f tanh, or with an activation t
// handed in the backward of that tanh, (x w)(1 - t^2).
//
// As library products of so few columns followed by element-wise passes these were ten launches a layer, of some ten
// microseconds of host time each, which is what a layer of a few hundred tokens waits for; here they are four (v6 layer T300
// H28: prefill 266 -> 233 us, forward+backward 922 -> 850).  On the GPU, 4096 rows of 4096 channels: 160 columns 60 + 5 ->
// 29 us, 64 columns 21 + 4 -> 22 forward and 51 + 4 -> 28 backward, the five planes 48 + 9 -> 64.  Bound by the latency of the
// reads of x, sixteen rows at a time (33 MB a plane: 7 us at the rate of a copy).
//
// A workgroup per 16 RT rows and plane, all columns: the rows are read once.  Its eight wavefronts share the contraction, 32
// deep in turn, two such steps in flight, and add up in LDS.  The weights (all of them per workgroup, from the L2) are the
// A operand: [column][k] straight from memory in the operand's layout, or, kept [k][column], in whole rows that are turned by
// the transposing LDS read.
#include "common.h"

namespace wkv {
namespace lora {

using rows::s8;
using rows::f4;
constexpr int WAVES = 8;

template <int NT, int RT, bool K_MAJOR> struct Tiles {
    static constexpr int LD = 16 * NT + 8;
    union {
        uint16_t w[K_MAJOR ? WAVES : 1][K_MAJOR ? 32 * LD : 8];          // a step's weights, rows in the order of w_row()
        f4 part[WAVES / 2][NT][RT][64];
    };
};
// where row k of a step goes, so that a lane's two transposing reads of four rows each hold eight consecutive k
__device__ __forceinline__ int w_row(int k) { return ((k >> 2) & 1) * 16 + (k >> 3) * 4 + (k & 3); }

template <int NT, int RT, bool K_MAJOR>
__global__ __launch_bounds__(64 * WAVES) void lora_down(int M, int K, const bf16 *__restrict__ x, const bf16 *__restrict__ w,
                                                        const bf16 *__restrict__ act, bf16 *__restrict__ out)
{
    typedef Tiles<NT, RT, K_MAJOR> Ti;
    extern __shared__ __align__(16) unsigned char raw[];
    Ti &sm = *reinterpret_cast<Ti *>(raw);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, n = lane & 15;
    const int row0 = 16 * RT * blockIdx.x, N = 16 * NT, ldo = N * gridDim.y;
    x += (size_t)blockIdx.y * M * K;
    w += (size_t)blockIdx.y * N * K;
    struct Step { s8 w[NT], x[RT]; };
    auto fetch = [&](Step &s, int k0) __attribute__((always_inline)) {
        k0 = min(k0, K - 32);          // (past the end: the last step again, unused)
#pragma unroll
        for (int i = 0; i < NT; i++) {
            const int p = lane + 64 * i;
            s.w[i] = K_MAJOR ? *reinterpret_cast<const s8 *>(w + (size_t)(k0 + p / (2 * NT)) * N + 8 * (p % (2 * NT)))
                             : *reinterpret_cast<const s8 *>(w + (size_t)(16 * i + n) * K + k0 + 8 * kg);
        }
#pragma unroll
        for (int i = 0; i < RT; i++) s.x[i] = *reinterpret_cast<const s8 *>(x + (size_t)min(row0 + 16 * i + n, M - 1) * K + k0 + 8 * kg);
    };
    f4 acc[NT][RT];
#pragma unroll
    for (int i = 0; i < NT; i++)
#pragma unroll
        for (int j = 0; j < RT; j++) acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const int tro = chunked::tr_lane_offset(lane, Ti::LD);
    auto use = [&](Step &s, int next) __attribute__((always_inline)) {
        s8 a[NT], b[RT];
#pragma unroll
        for (int j = 0; j < RT; j++) b[j] = s.x[j];
        if (K_MAJOR) {
            uint16_t *t = sm.w[wv];
            rows::wave_sync();
#pragma unroll
            for (int i = 0; i < NT; i++) {
                const int p = lane + 64 * i;
                *reinterpret_cast<s8 *>(t + w_row(p / (2 * NT)) * Ti::LD + 8 * (p % (2 * NT))) = s.w[i];
            }
            rows::wave_sync();
            fetch(s, next);
#pragma unroll
            for (int i = 0; i < NT; i++) {
                const chunked::s4 lo = chunked::frag_tr(t, tro + 16 * i), hi = chunked::frag_tr(t, tro + 16 * Ti::LD + 16 * i);
                a[i] = s8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
        } else {
#pragma unroll
            for (int i = 0; i < NT; i++) a[i] = s.w[i];
            fetch(s, next);
        }
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int j = 0; j < RT; j++) acc[i][j] = rows::mma(a[i], b[j], acc[i][j]);
    };
    // (Four steps in flight, whole lines of a row per wavefront, or workgroups that start at different places of the contraction
    // were each measured slower: 68 to 73 us against 64 for the five planes of 4096 rows, K 4096.)
    constexpr int STRIDE = 32 * WAVES;
    Step s0, s1;
    fetch(s0, 32 * wv);
    fetch(s1, 32 * wv + STRIDE);
    for (int k0 = 32 * wv; k0 < K; k0 += 2 * STRIDE) {
        use(s0, k0 + 2 * STRIDE);
        if (k0 + STRIDE < K) use(s1, k0 + 3 * STRIDE);
    }
    // the wavefronts' sums: the upper four hand theirs to the lower four, whose sums everybody adds up
    __syncthreads();
    if (wv >= WAVES / 2) {
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int j = 0; j < RT; j++) sm.part[wv - WAVES / 2][i][j][lane] = acc[i][j];
    }
    __syncthreads();
    if (wv < WAVES / 2) {
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int j = 0; j < RT; j++) sm.part[wv][i][j][lane] += acc[i][j];
    }
    __syncthreads();
    for (int tile = wv; tile < NT * RT; tile += WAVES) {
        const int i = tile / RT, j = tile % RT, m = row0 + 16 * j + n;
        const f4 s = (sm.part[0][i][j][lane] + sm.part[1][i][j][lane]) + (sm.part[2][i][j][lane] + sm.part[3][i][j][lane]);
        if (m >= M) continue;
        const size_t o = (size_t)m * ldo + blockIdx.y * N + 16 * i + 4 * kg;          // four consecutive columns of row m
        float y[4] = {s[0], s[1], s[2], s[3]};
        if (act) {
            float t[4];
            load4(act + o, t);
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] *= 1.f - t[e] * t[e];
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = tanhf(y[e]);
        }
        store4(out + o, y);
    }
}

template <int NT, int RT, bool K_MAJOR>
static hipError_t launch(hipStream_t s, int M, int K, int planes, const void *x, const void *w, const void *act, void *out) {
    constexpr size_t bytes = sizeof(Tiles<NT, RT, K_MAJOR>);
    static PerDevice lds_limit;
    const hipError_t e = lds_limit.once([] {
        return hipFuncSetAttribute((const void *)lora_down<NT, RT, K_MAJOR>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    });
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((lora_down<NT, RT, K_MAJOR>), dim3((M + 16 * RT - 1) / (16 * RT), planes), dim3(64 * WAVES), bytes, s, M, K,
                       (const bf16 *)x, (const bf16 *)w, (const bf16 *)act, (bf16 *)out);
    return hipGetLastError();
}
// 32 rows a workgroup halve what the workgroups read of the weights, 16 rows make twice as many of them
template <int NT, bool K_MAJOR>
static hipError_t launch(hipStream_t s, int M, int K, int planes, const void *x, const void *w, const void *act, void *out) {
    if ((M + 31) / 32 * planes < cu_count() / 2) return launch<NT, 1, K_MAJOR>(s, M, K, planes, x, w, act, out);
    return launch<NT, 2, K_MAJOR>(s, M, K, planes, x, w, act, out);
}
static bool lora_down_takes(int N, bool k_major) { return k_major ? N == 160 || N == 64 : N == 64 || N == 32; }
static hipError_t lora_down_launch(hipStream_t s, int M, int K, int N, int planes, bool k_major, const void *x, const void *w, const void *act, void *out) {
    if (k_major) return N == 160 ? launch<10, true>(s, M, K, planes, x, w, act, out) : launch<4, true>(s, M, K, planes, x, w, act, out);
    return N == 64 ? launch<4, false>(s, M, K, planes, x, w, act, out) : launch<2, false>(s, M, K, planes, x, w, act, out);
}

}  // namespace lora
}  // namespace wkv
