// The layer of a serving loop: one token per sequence, a few rows (sequences) at a time, bf16.  What a row costs is the
// weights, read once; as library products, element-wise passes and dtype conversions a v6 layer of one row was some 45
// launches (H32: 560 us, of which the weights need 22 us).  Here it is seven kernels, 46 us (47 with a walk over the jobs,
// the head's inputs and the last factor asked for where they are used, and barriers that wait for the new state to be written):
//
//   rows_products   any number of products  out = f(x' W)  of up to 64 rows with weights of their own, in one launch;
//                   x' may be the token-shift mix of x, formed where it is read (RWKV-v5/src/module/TimeMix.py:295-298,
//                   ChannelMix.py:46-47), and f one of the activations that follow a projection in a layer
//   lora_mix_rows   the five data-dependent mixes of the v6 TimeMix (RWKV-v6/src/module/TimeMix.py:264-276)
//   timemix_head    per head: the v6 decay's second LoRA product, the operator's single step, ln_x and the gate
//                   (RWKV-v6/src/module/TimeMix.py:280-298, RWKV-v5/src/module/TimeMix.py:309-320)
//
// Sums are fp32.  A result is rounded to bf16 wherever the layer's steps, run one by one (as the same layer with autograd
// on is), leave a tensor in memory: the mixed rows, the LoRAs' sums and their tanh, the raw decay, the operator's output, each
// projection before its activation.  So a token gives what it gives in a prompt or in training up to the order of sums.
// (Left in fp32 the layer's output differed by 5e-3 from the steps' and was no nearer to 64 bits: 5.4e-3 against 5.6e-3.)
#include "common.h"

namespace wkv {
namespace rows {

typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int MAX_ROWS = 64, MAX_JOBS = 8;
struct Job {
    const bf16 *w;          // [N][K], k_major: [K][N]
    const bf16 *x;          // [rows][K]
    const bf16 *shift;      // [rows][K], with mix
    const bf16 *mix;        // [K], or NULL: x as it is
    const bf16 *mul;        // [rows][N], ACT_SIGMOID_MUL
    void *out;              // bf16 [rows][N]; k_major: fp32 [SPLIT][rows][N], parts of the sum
    int n, k_major, lerp, act;
};
// end[i]: the workgroups of jobs 0 .. i, past the last job INT_MAX.  A workgroup finds its job by one scalar load of all of
// them; a walk over the jobs is a scalar load and its latency for each.
struct Jobs { Job j[MAX_JOBS]; int end[MAX_JOBS], count; };
static_assert(MAX_JOBS == 8, "");
enum { ACT_NONE = 0, ACT_RELU_SQUARE = 1, ACT_SIGMOID_MUL = 2 };

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

// A workgroup per TN columns (8, 16 or 32); its wavefronts share the contraction and meet in LDS.  The weights are the A
// operand of the MFMAs (their columns are the rows there), the rows of x the B operand: lane (kg = lane/16, n = lane%16)
// supplies weight row n and x row n, eight consecutive k each.
//
// Bound by the weights, so by how they are fetched.  Read in the operand's own layout (16 rows x 64 bytes an instruction)
// a layer's weights come at 3.4 TB/s; read along the rows, at up to 4.  So a wavefront takes TN rows x SEG = 4096 / TN k
// at a time that way into registers (two such segments in flight, used in turn, where XL leaves the registers) and turns them in
// LDS that belongs to it alone; the same for the rows of x, of which only those that exist are read, and mixed on the way.
//
// XL fetches of x, each 512 elements: one row of a segment of 512 k (TN 8), two of 256 (TN 16) or four of 128 (TN 32).
template <int TN, int XL> struct Shape {
    static constexpr int SEG = 4096 / TN, LD = SEG + 8, PER = TN / 8;     // k of a segment, padded row in LDS, rows per fetch
    static constexpr int XROWS = PER * XL, MT = (XROWS + 15) / 16, NT = (TN + 15) / 16;      // MFMA tiles of rows, of columns
    static __device__ int row(int lane) { return lane / (SEG / 8); }
    static __device__ int k(int lane) { return 8 * (lane % (SEG / 8)); }
};
template <int TN, int XL> struct Turn { uint16_t w[TN * Shape<TN, XL>::LD], x[Shape<TN, XL>::XROWS * Shape<TN, XL>::LD]; };

template <int XL, bool MIX> struct Segment { s8 w[8], x[XL], shift[MIX ? XL : 1], mix; };
template <int TN, int XL, bool MIX>
__device__ __forceinline__ void fetch(Segment<XL, MIX> &s, const Job &job, const bf16 *w, int row0, int rows, int K, int k0, int lane) {
    typedef Shape<TN, XL> Sh;
    const int k = min(k0 + Sh::k(lane), K - 8);              // (past the end: read again and not used)
#pragma unroll
    for (int i = 0; i < 8; i++) s.w[i] = *reinterpret_cast<const s8 *>(w + (size_t)(Sh::PER * i) * K + k);
#pragma unroll
    for (int i = 0; i < XL; i++)
        if (row0 + Sh::PER * i < rows) {
            const size_t o = (size_t)min(row0 + Sh::PER * i + Sh::row(lane), rows - 1) * K + k;
            s.x[i] = *reinterpret_cast<const s8 *>(job.x + o);
            if (MIX) s.shift[i] = *reinterpret_cast<const s8 *>(job.shift + o);
        }
    if (MIX) s.mix = *reinterpret_cast<const s8 *>(job.mix + k);
}
template <int TN, int XL, bool MIX>
__device__ __forceinline__ void turn(const Segment<XL, MIX> &s, Turn<TN, XL> &t, const Job &job, int row0, int rows, int lane) {
    typedef Shape<TN, XL> Sh;
    const int o = Sh::row(lane) * Sh::LD + Sh::k(lane);
#pragma unroll
    for (int i = 0; i < 8; i++) *reinterpret_cast<s8 *>(&t.w[Sh::PER * i * Sh::LD + o]) = s.w[i];
#pragma unroll
    for (int i = 0; i < XL; i++)
        if (row0 + Sh::PER * i < rows)
            *reinterpret_cast<s8 *>(&t.x[Sh::PER * i * Sh::LD + o]) = MIX ? mixed(s.x[i], s.shift[MIX ? i : 0], s.mix, job.lerp) : s.x[i];
}
// (lanes whose row of x does not exist repeat the last one, and those beyond 8 weight rows repeat them: rows and columns
// of the result that nobody reads)
template <int TN, int XL>
__device__ __forceinline__ void multiply(const Turn<TN, XL> &t, int steps, int live, int lane, f4 (&acc)[Shape<TN, XL>::NT][Shape<TN, XL>::MT]) {
    typedef Shape<TN, XL> Sh;
    const int n = lane & 15, k = 8 * (lane >> 4);
    int xo[Sh::MT];
#pragma unroll
    for (int mt = 0; mt < Sh::MT; mt++) xo[mt] = min(16 * mt + n, live - 1) * Sh::LD + k;
#pragma unroll
    for (int i = 0; i < Sh::SEG / 32; i++)
        if (i < steps) {
            s8 a[Sh::NT];
#pragma unroll
            for (int nt = 0; nt < Sh::NT; nt++) a[nt] = *reinterpret_cast<const s8 *>(&t.w[(16 * nt + n % TN) * Sh::LD + k + 32 * i]);
#pragma unroll
            for (int mt = 0; mt < Sh::MT; mt++) {
                const s8 x = *reinterpret_cast<const s8 *>(&t.x[xo[mt] + 32 * i]);
#pragma unroll
                for (int nt = 0; nt < Sh::NT; nt++) acc[nt][mt] = mma(a[nt], x, acc[nt][mt]);
            }
        }
}
// the lanes of a wavefront exchange data through LDS: program order is enough for the hardware, the compiler is told
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int TN, int XL, int WAVES, bool MIX>
__device__ __forceinline__ void accumulate(const Job &job, Turn<TN, XL> &t, int tile, int row0, int rows, int K, int wv, int lane,
                                           f4 (&acc)[Shape<TN, XL>::NT][Shape<TN, XL>::MT]) {
    typedef Shape<TN, XL> Sh;
    constexpr bool TWO = XL <= 8;                            // two segments in flight where the registers allow it
    const bf16 *w = job.w + (size_t)(TN * tile + Sh::row(lane)) * K;
    const int step = WAVES * Sh::SEG, live = min(rows - row0, Sh::XROWS);
    Segment<XL, MIX> a, b;
    auto use = [&](Segment<XL, MIX> &s, int k0, int ahead) __attribute__((always_inline)) {
        wave_sync();
        turn<TN>(s, t, job, row0, rows, lane);
        if (k0 + ahead < K) fetch<TN>(s, job, w, row0, rows, K, k0 + ahead, lane);
        wave_sync();
        multiply(t, min(Sh::SEG, K - k0) / 32, live, lane, acc);
    };
    const int first = wv * Sh::SEG;
    if (first >= K) return;
    fetch<TN>(a, job, w, row0, rows, K, first, lane);
    if (TWO && first + step < K) fetch<TN>(b, job, w, row0, rows, K, first + step, lane);
    for (int k0 = first; k0 < K; k0 += (TWO ? 2 : 1) * step) {
        use(a, k0, (TWO ? 2 : 1) * step);
        if (TWO && k0 + step < K) use(b, k0 + step, 2 * step);
    }
}
// The weights of the LoRAs are kept [k][n]: two bytes at a time in the operand's layout.  Their columns are few (160 and
// 64), so the contraction is cut into SPLIT parts for workgroups of their own (10 workgroups took 6.6 us for the 160
// columns of a row at K 2048); whoever reads the result adds the parts.
constexpr int SPLIT = 8;
template <int MT, int WAVES, bool MIX>
__device__ __forceinline__ void accumulate_k_major(const Job &job, int tile, int part, int row0, int rows, int K, int wv, int lane, f4 (&acc)[MT]) {
    const int kg = lane >> 4, n = lane & 15, last = (part + 1) * (K / 32) / SPLIT;
    for (int step = part * (K / 32) / SPLIT + wv; step < last; step += WAVES) {
        const int k = 32 * step + 8 * kg;
        s8 a;
        const bf16 *w = job.w + (size_t)k * job.n + 16 * tile + n;
#pragma unroll
        for (int e = 0; e < 8; e++) a[e] = (short)w[(size_t)e * job.n].bits;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const size_t o = (size_t)min(row0 + 16 * mt + n, rows - 1) * K + k;
            const s8 x = *reinterpret_cast<const s8 *>(job.x + o);
            acc[mt] = mma(a, MIX ? mixed(x, *reinterpret_cast<const s8 *>(job.shift + o), *reinterpret_cast<const s8 *>(job.mix + k), job.lerp) : x, acc[mt]);
        }
    }
}

template <int TN> __host__ __device__ inline int workgroups(const Job &job) { return job.k_major ? job.n / 16 * SPLIT : job.n / TN; }

template <int TN, int XL, int WAVES>
__global__ __launch_bounds__(64 * WAVES, XL <= 2 ? 4 : 2) void rows_products(int rows, int K, Jobs jobs) {
    constexpr int MT = Shape<TN, XL>::MT, NT = Shape<TN, XL>::NT;
    __shared__ __align__(16) Turn<TN, XL> turned[WAVES];
    // a wavefront's sums go where it turned its own weights, so that no other has to be done with them
    auto part = [&](int wave, int tile) __attribute__((always_inline)) { return reinterpret_cast<f4 *>(&turned[wave]) + tile * 64; };
    static_assert(sizeof(turned[0]) % sizeof(f4) == 0, "");
    static_assert(sizeof(turned[0]) >= NT * MT * 64 * sizeof(f4), "the sums fit where the weights were turned");
    int ji = 0, before = 0;
    const int row0 = Shape<TN, XL>::XROWS * blockIdx.y;
#pragma unroll
    for (int i = 0; i < MAX_JOBS - 1; i++)                   // (the grid is the sum over all jobs)
        if ((int)blockIdx.x >= jobs.end[i]) { ji = i + 1; before = jobs.end[i]; }
    const int wg = blockIdx.x - before;
    const Job job = jobs.j[ji];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kg = lane >> 4, n = lane & 15;
    // the lane holds four consecutive columns of row m of a tile
    auto row_of = [&](int tile) { return row0 + 16 * (tile % MT) + n; };
    auto at = [&](int tile) { return (size_t)row_of(tile) * job.n + TN * wg + 16 * (tile / MT) + 4 * kg; };
    auto mine = [&](int tile) { return tile < NT * MT && row_of(tile) < rows && (TN > 8 || kg < 2); };
    uint2 factor = make_uint2(0u, 0u);                       // asked for before the weights, not behind the sums
    if (job.act == ACT_SIGMOID_MUL && !job.k_major && mine(wv)) factor = *reinterpret_cast<const uint2 *>(job.mul + at(wv));
    f4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[nt][mt] = f4{0.f, 0.f, 0.f, 0.f};
    if (job.k_major) {
        if (job.mix) accumulate_k_major<MT, WAVES, true>(job, wg / SPLIT, wg % SPLIT, row0, rows, K, wv, lane, acc[0]);
        else accumulate_k_major<MT, WAVES, false>(job, wg / SPLIT, wg % SPLIT, row0, rows, K, wv, lane, acc[0]);
    } else {
        if (job.mix) accumulate<TN, XL, WAVES, true>(job, turned[wv], wg, row0, rows, K, wv, lane, acc);
        else accumulate<TN, XL, WAVES, false>(job, turned[wv], wg, row0, rows, K, wv, lane, acc);
    }
    wave_sync();
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) part(wv, nt * MT + mt)[lane] = acc[nt][mt];
    lds_barrier();
    for (int tile = wv; tile < (job.k_major ? 1 : NT) * MT; tile += WAVES) {
        f4 s = part(0, tile)[lane];
#pragma unroll
        for (int i = 1; i < WAVES; i++) s += part(i, tile)[lane];
        const int m = row_of(tile);
        if (m >= rows) continue;
        float y[4] = {s[0], s[1], s[2], s[3]};
        if (job.k_major) {
            store4((float *)job.out + ((size_t)(wg % SPLIT) * rows + m) * job.n + 16 * (wg / SPLIT) + 4 * kg, y);
            continue;
        }
        if (TN == 8 && kg >= 2) continue;
        const size_t o = at(tile);
        if (job.act == ACT_RELU_SQUARE) {
#pragma unroll
            for (int e = 0; e < 4; e++) { const float p = fmaxf(round_bf16(y[e]), 0.f); y[e] = p * p; }
        } else if (job.act == ACT_SIGMOID_MUL) {
            if (tile != wv) factor = *reinterpret_cast<const uint2 *>(job.mul + o);
            const float q[4] = {bf((uint16_t)factor.x), bf((uint16_t)(factor.x >> 16)), bf((uint16_t)factor.y), bf((uint16_t)(factor.y >> 16))};
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = sigmoid(q[e]) * round_bf16(y[e]);
        }
        store4((bf16 *)job.out + o, y);
    }
}

// out[j] = x + (shift - x) (maa_j + act_j w2_j): a wavefront per mix and 16 channels, whose 32-deep product is one MFMA
// per 16 rows.  act [SPLIT][rows][5][32], parts of the first LoRA product, whose tanh is taken here; w2 [5][32][C].
struct Maa { const bf16 *p[5]; };
__global__ __launch_bounds__(320) void lora_mix_rows(int rows, int C, const bf16 *__restrict__ x, const bf16 *__restrict__ shift,
        Maa maa, const float *__restrict__ act, const bf16 *__restrict__ w2, bf16 *__restrict__ out)
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
        const size_t o = (size_t)mc * C + c0 + 4 * kg;
        float xv[4], xx[4], y[4];
        load4(x + o, xv);
        load4(shift + o, xx);
        float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < SPLIT; p++) {
            const float *q = act + (((size_t)p * rows + mc) * 5 + j) * 32 + 8 * kg;
            const float4 lo = *reinterpret_cast<const float4 *>(q), hi = *reinterpret_cast<const float4 *>(q + 4);
            t[0] += lo.x; t[1] += lo.y; t[2] += lo.z; t[3] += lo.w;
            t[4] += hi.x; t[5] += hi.y; t[6] += hi.z; t[7] += hi.w;
        }
#pragma unroll
        for (int e = 0; e < 8; e++) t[e] = tanhf(round_bf16(t[e]));
        const uint4 bp = make_uint4(bf16_pack2(t[0], t[1]), bf16_pack2(t[2], t[3]), bf16_pack2(t[4], t[5]), bf16_pack2(t[6], t[7]));
        const s8 b = __builtin_bit_cast(s8, bp);
        const f4 dyn = mma(a, b, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = fmaf(xx[e] - xv[e], d[e] + dyn[e], xv[e]);
        if (m < rows) store4(out + (size_t)j * rows * C + o, y);
    }
}

// One workgroup per (row, head), lane (key group, four value columns) as in decode56.  lora != NULL (v6): the raw decay
// of the head's channels is time_decay + tanh(lora[row]) w2 (64 deep), lora [SPLIT][rows][64] in parts; NULL (v5): time_decay itself.
__global__ __launch_bounds__(256) void timemix_head(int H, const bf16 *__restrict__ r, const bf16 *__restrict__ k, const bf16 *__restrict__ v,
        const bf16 *__restrict__ gate, const bf16 *__restrict__ time_decay, const float *__restrict__ lora, const bf16 *__restrict__ w2,
        const bf16 *__restrict__ u, const bf16 *__restrict__ ln_w, const bf16 *__restrict__ ln_b, float scale, float eps,
        const float *s_in, float *s_out, bf16 *__restrict__ out)
{
    __shared__ __align__(16) float part[4][HEAD], dec[HEAD];
    const int row = blockIdx.x / H, h = blockIdx.x % H, C = H * HEAD, tid = threadIdx.x, kq = tid >> 4, c4 = 4 * (tid & 15);
    const size_t base = (size_t)row * C + h * HEAD, so = (size_t)blockIdx.x * HEAD * HEAD;
    // Latency, one round trip to memory after another: everything is asked for here, and no barrier waits for the state
    // to be written.
    float4 S[4];
    bf16 rb[4], kb[4], ub[4];
    uint2 vb = *reinterpret_cast<const uint2 *>(v + base + c4);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int key = kq + 16 * i;
        rb[i] = r[base + key]; kb[i] = k[base + key]; ub[i] = u[h * HEAD + key];
        S[i] = *reinterpret_cast<const float4 *>(s_in + so + key * HEAD + c4);
    }
    const int own = h * HEAD + (tid & 63);
    const float decay_own = to_float(time_decay[own]), g = to_float(gate[base + (tid & 63)]);
    const float lnw = to_float(ln_w[own]), lnb = to_float(ln_b[own]);
    {
        const int ch = tid & 63, q = tid >> 6;
        float a = 0.f, w2v[16];
        if (lora) {
#pragma unroll
            for (int e = 0; e < 16; e++) w2v[e] = to_float(w2[(size_t)(16 * q + e) * C + h * HEAD + ch]);
            if (tid < HEAD) {
                float t = 0.f;
#pragma unroll
                for (int p = 0; p < SPLIT; p++) t += lora[((size_t)p * (gridDim.x / H) + row) * HEAD + tid];
                dec[tid] = round_bf16(tanhf(round_bf16(t)));
            }
            lds_barrier();
#pragma unroll
            for (int e = 0; e < 16; e++) a = fmaf(dec[16 * q + e], w2v[e], a);
        }
        part[q][ch] = a;
        lds_barrier();
        if (tid < HEAD)
            dec[tid] = __expf(log_decay(round_bf16(decay_own + ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]))), false));
        lds_barrier();
    }
    const float v4[4] = {bf((uint16_t)vb.x), bf((uint16_t)(vb.x >> 16)), bf((uint16_t)vb.y), bf((uint16_t)(vb.y >> 16))};
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, bonus = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int key = kq + 16 * i;
        const float ri = to_float(rb[i]), ki = to_float(kb[i]), wi = dec[key];
        bonus = fmaf(ri * to_float(ub[i]), ki, bonus);
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
    lds_barrier();
    if (tid >= HEAD) return;
    const float y = scale * round_bf16((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]));
    float s = y;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
    const float dy = y - s * (1.f / HEAD);
    float q = dy * dy;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) q += __shfl_xor(q, o);
    const float z = fmaf(dy * rsqrtf(q * (1.f / HEAD) + eps), lnw, lnb);
    out[base + tid] = from_float<bf16>(z * g * sigmoid(g));
}

// Which shape.  Every workgroup reads all the rows of x for its columns, so from three rows on that traffic, and the mixing,
// is of the weights' size with 16 columns; 32 columns halve it for half as many workgroups.  v6 layer, 16 -> 32 columns in
// us: 20 rows H40 97.6 -> 80.7, 64 rows H40 203 -> 158, 64 rows H64 389 -> 289, 16 rows H28 50.7 -> 45.3.  Up to 16 rows they pay
// where the workgroups still reach most compute units and not yet all of them twice (H64, 544 workgroups: 140 us with 16
// columns, 154 with 32; its output projection, 128: 256 of 16 columns are 5 % faster); from 33 rows on, where 16 columns
// read the weights twice, once half the compute units have one (H12: 56 against 61 us); between, down to 32 workgroups.
// One or two rows: 8 columns where 16 would leave compute units idle.  Eight wavefronts where the workgroups do not fill
// the compute units twice over, four (of which several workgroups share a compute unit) otherwise.
static hipError_t rows_products_launch(hipStream_t s, int rows, int K, Jobs &jobs) {
    int wgs32 = 0, wgs16 = 0, wgs8 = 0;
    bool by32 = true;
    for (int i = 0; i < jobs.count; i++) {
        wgs32 += workgroups<32>(jobs.j[i]); wgs16 += workgroups<16>(jobs.j[i]); wgs8 += workgroups<8>(jobs.j[i]);
        by32 = by32 && (jobs.j[i].k_major || jobs.j[i].n % 32 == 0);
    }
    auto total = [&](auto columns) {
        int sum = 0;
        for (int i = 0; i < MAX_JOBS; i++) {
            if (i < jobs.count) sum += workgroups<decltype(columns)::value>(jobs.j[i]);
            jobs.end[i] = i < jobs.count ? sum : INT_MAX;
        }
    };
#define WKV_ROWS(TN, XL, WAVES)                                                                                        \
    do {                                                                                                               \
        total(std::integral_constant<int, TN>());                                                                      \
        hipLaunchKernelGGL((rows_products<TN, XL, WAVES>), dim3(TN == 32 ? wgs32 : TN == 16 ? wgs16 : wgs8, (rows + TN * XL / 8 - 1) / (TN * XL / 8)), \
                           dim3(64 * WAVES), 0, s, rows, K, jobs);                                                      \
    } while (0)
    const int ncu = cu_count();
    if (rows > 32) { if (by32 && wgs32 > ncu / 2) WKV_ROWS(32, 16, 4); else WKV_ROWS(16, 16, 4); }
    else if (rows > 16) {
        if (!by32 || wgs32 < ncu / 8) WKV_ROWS(16, 16, 4);
        else if (wgs32 < 2 * ncu) WKV_ROWS(32, 8, 8);
        else WKV_ROWS(32, 8, 4);
    } else if (rows > 2) {
        if (by32 && wgs32 > ncu / 2 && wgs32 < 2 * ncu) { if (wgs32 < ncu) WKV_ROWS(32, 4, 8); else WKV_ROWS(32, 4, 4); }
        else if (wgs16 < 2 * ncu) WKV_ROWS(16, 8, 8);
        else WKV_ROWS(16, 8, 4);
    }
    else if (wgs16 < ncu) WKV_ROWS(8, 2, 8);
    else if (wgs16 < 2 * ncu) WKV_ROWS(16, 1, 8);
    else WKV_ROWS(16, 1, 4);
#undef WKV_ROWS
    return hipGetLastError();
}

}  // namespace rows
}  // namespace wkv
