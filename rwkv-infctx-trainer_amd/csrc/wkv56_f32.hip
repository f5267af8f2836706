// WKV5 / WKV6 in blocked form with fp32 products: fp32 and fp16 streams with the decay floor, sequences long enough for
// 64-token steps to pay (steps_pay in api.hip; wkv56_chunked.hip is the same for bf16 streams, whose operands it splits
// into bf16 parts).
//
// The token-by-token kernels (wkv56_recurrent.hip) walk the tokens one after another at 4096 multiply-adds a head and
// token forward, four times that backward, on the vector pipe: B8 T4096 H40 fp32 4.05 ms forward and backward, and a
// short batch leaves most of the chip idle for as long as its tokens last.  Here the same fp32 multiply-adds are
// v_mfma_f32_16x16x4_f32 (twice the vector pipe's rate, operands shared by 16 lanes), 16 tokens at a time, and a
// sequence is cut into time segments as in the bf16 kernels.
//
// Blocks of 16 tokens with exponents counted from the block's MIDDLE: with m the sum of log w over the block's first
// eight tokens, b over all of it, and for token t  x_t = (sum over the tokens before t) - m,
//
//     rm_t = r_t e^{x_t},   km_t = k_t e^{-(x_t + log w_t)},   S1 = e^{m} o S
//     y_t  = rm_t S1 + sum_{s<t} (rm_t . km_s) v_s + (r_t . u k_t) v_t
//     S   <- e^{b-m} o (S1 + sum_s km_s^T v_s)
//
// so one scaled copy of r and of k serves every product, and with the 0.005 floor no exponent leaves +-43 (the sums over
// half a block; the block's start as origin would need twice that).  Backward, with G the gradient of the state at the
// block's end, G1 = e^{b-m} o G and P[t][s] = gy_t . v_s:
//
//     d(rm)_t = S1 gy_t + sum_{s<t} P[t][s] km_s        gr_t = e^{x_t} d(rm)_t + u k_t P[t][t]
//     d(km)_s = G1 v_s  + sum_{t>s} P[t][s] rm_t        gk_s = e^{-(x_s + log w_s)} d(km)_s + u r_s P[s][s]
//     gv_s    = km_s G1 + sum_{t>s} (rm_t . km_s) gy_t + (r_s . u k_s) gy_s
//     G      <- e^{m} o (G1 + sum_t rm_t^T gy_t)
//
// and the decay gradient from the running sum  A_{t-1} = A_t + rm_t d(rm)_t - km_t d(km)_t  (the bonus terms cancel),
// dL/dlog w_t = A_t - km_t d(km)_t.  The bonus terms come from the scaled copies too: u k_t P = e^{x_t} (u w_t km_t P),
// u r_t P = e^{-(x_t + log w_t)} (u w_t rm_t P).
//
// Non-finite and very large values.  The masked products multiply zeros with what a later (backward: an earlier) token of the
// block holds, which an infinity or a NaN turns into NaN, and the scaled copies and their products reach 2^61 times the values:
// a token's past would not stay clean of it, and some results would overflow that fit.  So a step that holds a NaN, an
// infinity or anything beyond 2^18 (found where it is prepared) is walked token by token by the wavefronts that own the
// states, in the recurrence's own terms.  Up to that bound no product of the blocked form overflows: 16 tokens x 64 values x
// 2^(18+18) x 2^(61.2+18) < 2^126.  The check costs 0 to 2 % of a forward; B8 T2048 H40 fp32, forward and backward, without it
// 722 us (WKV5) and 800 us (WKV6), with it 749 and 774.  What the state holds, an infinity too, is carried from step to step as the
// recurrence carries it; between time segments it is forgotten once its decay has left 2^-PASS_CUT of it, like anything else.
//
// Operand layouts (lane = 16 g + n): A[m = n][k = 4 g' .. ] and B[k][n], where the k of a 16-deep product may be dealt out
// in any order; taken as k = 4 g + e for the e-th of four instructions, the operand read along its rows is one 16-byte LDS
// read, the one read along its columns four 4-byte ones, and a result tile (rows 4 g + e, column n) is at once the
// operand of a product over its rows: states and masked matrices go from accumulator to operand as they are.
#include "common.h"

namespace wkv {
namespace f32 {

using chunked::PART;
using chunked::SB;
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int LD = chunked::CHAIN_LD;      // padded rows of a [64][64] table: conflict-free along rows and along columns
constexpr int NT = 512;       // eight wavefronts

__device__ __forceinline__ f4 zero4() { return f4{0.f, 0.f, 0.f, 0.f}; }
__device__ __forceinline__ f4 mma(f4 a, f4 b, f4 c) {          // a 16-deep product
#pragma unroll
    for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
}
__device__ __forceinline__ f4 along(const float *t, int row, int col) { return *reinterpret_cast<const f4 *>(t + row * LD + col); }      // [row][col..col+3]
__device__ __forceinline__ f4 across(const float *t, int row, int col) {                                                              // [row..row+3][col]
    return f4{t[row * LD + col], t[(row + 1) * LD + col], t[(row + 2) * LD + col], t[(row + 3) * LD + col]};
}
// the lanes of a wavefront exchange data through LDS: program order is enough for the hardware, the compiler is told
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// element `o` of the row of token t (the same for all lanes): scalar base + 32-bit lane offset
template <class P> __device__ __forceinline__ P *row_at(P *p, int t, int C, uint32_t o) { return chunked::seq_at(p + (size_t)t * C, o); }

// Results leave by buffer stores, which drop what lies beyond the sequence's end: no branch around them, so that the
// compiler can count them and a wait for loads issued before them does not wait for the stores too (loads and stores
// share one counter, and after a store that may or may not have been issued it waits for everything outstanding).
// `left`: elements from `p` to the end of the sequence.  The whole offset goes through the lane's register: only that is
// compared with the end without wrapping (and the API sends sequences within 64 rows of 2^32 bytes another way).
struct Out { __amdgpu_buffer_rsrc_t rsrc; };
template <class P> __device__ __forceinline__ Out out_of(P *p, size_t left) {
    return Out{__builtin_amdgcn_make_buffer_rsrc(const_cast<void *>((const void *)p), (short)0, (int)(uint32_t)(left * sizeof(P)), 0x00027000)};
}
// element lane_o of row t (uniform)
template <class P> __device__ __forceinline__ void put(const Out &o, int t, int C, uint32_t lane_o, float x) {
    const P v = from_float<P>(x);
    const int vo = (int)(((uint32_t)t * C + lane_o) * sizeof(P));
    if constexpr (sizeof(P) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), o.rsrc, vo, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, v), o.rsrc, vo, 0, 0);
}
template <class P> __device__ __forceinline__ void put4(const Out &o, int t, int C, uint32_t lane_o, f4 x) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const int vo = (int)(((uint32_t)t * C + lane_o) * sizeof(P));
    if constexpr (sizeof(P) == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, x), o.rsrc, vo, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, h4{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]}), o.rsrc, vo, 0, 0);
}

// Preparation of N consecutive tokens of one channel per lane.  x[i] as above for tokens counted from the block's middle:
// the tokens before it (LATE = false) sum backwards from it, those after it forwards.
template <int N, bool LATE>
__device__ __forceinline__ float half_exponents(const float (&lw)[N], float (&x)[N]) {
    float s = 0.f;
    if (LATE) {
#pragma unroll
        for (int i = 0; i < N; i++) { x[i] = s; s += lw[i]; }
    } else {
#pragma unroll
        for (int i = N - 1; i >= 0; i--) { s += lw[i]; x[i] = -s; }
    }
    return s;          // log2 of the half's decay
}
// sums over the 64 lanes of eight per-token values, left as the four partial sums of the lane groups: part[group][token]
__device__ __forceinline__ void store_row_sums(const float (&p)[8], float (*part)[8], int lane) {
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; i++) s[i] = chunked::row_prefix_sum(p[i]);
    if ((lane & 15) == 15) {
        *reinterpret_cast<f4 *>(&part[lane >> 4][0]) = f4{s[0], s[1], s[2], s[3]};
        *reinterpret_cast<f4 *>(&part[lane >> 4][4]) = f4{s[4], s[5], s[6], s[7]};
    }
}
__device__ __forceinline__ float row_sum(const float (*part)[4][8], int tok) {       // part[half block][group][token]
    const float (*p)[8] = part[tok >> 3];
    return (p[0][tok & 7] + p[1][tok & 7]) + (p[2][tok & 7] + p[3][tok & 7]);
}

// the largest absolute value, NaN if there is one (one v_maximum3_f32)
__device__ __forceinline__ float largest(float m, float a, float b) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, fabsf(a)), fabsf(b));
}
constexpr float PLAIN_LIMIT = 262144.f;      // 2^18
__device__ __forceinline__ void store_plain(int *plain, float m, int lane) {          // m: of the wavefront's eight tokens, per channel
    const bool any = __builtin_amdgcn_ballot_w64(!(m <= PLAIN_LIMIT)) != 0;
    if (lane == 0) *plain = any;
}
__device__ __forceinline__ int any_plain(const int (&plain)[8]) {
    const int4 a = *reinterpret_cast<const int4 *>(&plain[0]), b = *reinterpret_cast<const int4 *>(&plain[4]);
    return (a.x | a.y) | (a.z | a.w) | (b.x | b.y) | (b.z | b.w);
}
__device__ __forceinline__ bool rarely(int x) { return __builtin_expect(__builtin_amdgcn_readfirstlane(x) != 0, 0); }      // the same in all lanes
__device__ __forceinline__ float over_groups(float x) {          // over the four lane groups, in every lane
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}

// ------------------------------------------------------------------------------------------------------------ forward --
// Twelve wavefronts, one barrier per 64-token step.  Wavefronts 0-3 walk the state (values 16 w .. +15, all keys) over
// the step's four blocks.  Wavefronts 4-11 meanwhile build the masked matrices of the step and prepare half a block each
// of the NEXT step in the other buffer; after the barrier the first four add the matrices' products to the y they hold
// in registers.  Bound by the matrix pipe: 160 instructions of 32 clocks per SIMD and step.  (With the eight wavefronts
// that fill two per SIMD, a whole block's preparation per wavefront took 12 k clocks a step, the walk 7 k.)
constexpr int NT_FWD = 768;
// Who walks the piece summaries before a segment: the four wavefronts that own the state, while the others prepare the first
// step, or, where there are more pieces than this and a decay that forgets nothing may have to walk them all, eight wavefronts
// with half as many loads each, four of which prepare afterwards.  Prompts, four / eight wavefronts / by this rule, us: fp32
// H4 T300 (4 pieces) 14.8 / 15.5 / 14.4, H12 T777 (12) 18.4 / 19.1 / 18.1, H32 T2048 47.0 / 47.7 / 45.7; H4 T2048 (31) 22.1 / 22.0 /
// 21.0, H4 T4096 (63) 36.6 / 32.0 / 30.4; with a decay that forgets within a piece, H4 T4096, 21.2 / 20.8 / 20.9.  (The third
// figures are also without the second step's inputs asked for during the walk.)
constexpr int LONG_WALK = 16;
struct FwdTiles {
    float rm[SB * LD], km[SB * LD], v[SB * LD];
    float em[4][HEAD], eb[4][HEAD];      // e^{m}, e^{b-m} per block and key
    float rho[8][4][8];                  // r . (u o k) per token, in parts
    alignas(16) int plain[8];            // half a block each: the step is walked token by token
};
struct FwdShared {
    FwdTiles step[2];
    f4 at[2][4][64];                     // masked matrix of each block of a step: rows s, columns t
};

template <class T, class W, bool PER_TOKEN_W>
__global__ __launch_bounds__(NT_FWD) void forward_f32(int bh0, int Tlen, int C, int H, int nseg, int sps, int m,
        const T *__restrict__ r, const T *__restrict__ k, const T *__restrict__ v, const W *__restrict__ wraw,
        const float *__restrict__ u, const float *s_in, T *__restrict__ y, float *s_out, float *__restrict__ ckpt,
        const float *__restrict__ part, int floor_decay)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    FwdShared &sh = *reinterpret_cast<FwdShared *>(smem_raw);
    const int bh = bh0 + blockIdx.x / nseg, seg = blockIdx.x % nseg, b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, w8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, n = lane & 15;
    const bool chain = w8 < 4;
    const int q = chain ? w8 : (w8 - 4) >> 1, hf = w8 & 1;      // value quarter; block and half of it
    {
        const size_t base = (size_t)b * Tlen * C + (size_t)h * HEAD;
        r += base; k += base; v += base;
        if (y) y += base;
        if (PER_TOKEN_W) wraw += base;
    }
    const int nsb = (Tlen + SB - 1) / SB, sb0 = seg * sps, sb1 = min(nsb, (seg + 1) * sps);

    // preparing wavefronts: tokens tok0 .. tok0+7 of the step, channel `lane`
    const int tok0 = 16 * q + 8 * hf;
    const float uf = u[h * HEAD + lane];
    const float l_const = PER_TOKEN_W ? 0.f : log2_decay(to_float(wraw[h * HEAD + lane]), floor_decay);
    T tr[8], tk[8], tv[8];
    W tw[8];
    auto fetch = [&](int sb) __attribute__((always_inline)) {          // (tokens past the end are read from the last one and replaced)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int t = min(sb * SB + tok0 + i, Tlen - 1);
            tr[i] = *row_at(r, t, C, lane); tk[i] = *row_at(k, t, C, lane); tv[i] = *row_at(v, t, C, lane);
            if (PER_TOKEN_W) tw[i] = *row_at(wraw, t, C, lane);
        }
    };
    auto prepare = [&](int sb, FwdTiles &sm) __attribute__((always_inline)) {
        float lw[8], x[8], p[8], m = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++)
            lw[i] = sb * SB + tok0 + i >= Tlen ? 0.f : PER_TOKEN_W ? log2_decay(to_float(tw[i]), floor_decay) : l_const;
        const float total = hf ? half_exponents<8, true>(lw, x) : half_exponents<8, false>(lw, x);
        (hf ? sm.eb : sm.em)[q][lane] = exp2_fast(total);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const bool in = sb * SB + tok0 + i < Tlen;
            const float rf = in ? to_float(tr[i]) : 0.f, kf = in ? to_float(tk[i]) : 0.f, vf = in ? to_float(tv[i]) : 0.f;
            const int o = (tok0 + i) * LD + lane;
            sm.rm[o] = rf * exp2_fast(x[i]);
            sm.km[o] = kf * exp2_fast(-(x[i] + lw[i]));
            sm.v[o] = vf;
            p[i] = rf * uf * kf;
            m = largest(m, rf, kf);
            m = largest(m, vf, PER_TOKEN_W ? lw[i] : vf);
        }
        store_row_sums(p, sm.rho[2 * q + hf], lane);
        store_plain(&sm.plain[2 * q + hf], m, lane);
    };
    const float *sp = s_in + (size_t)bh * HEAD * HEAD;
    const float *pieces = part + (size_t)bh * nseg * m * PART;
    float *table = sh.step[1].rm;                // the state at the segment's start (not in use yet)
    const bool long_walk = seg * m > LONG_WALK;
    // (the two roles have loops of their own: in a common one the compiler waits, in either, for what the other may have
    // outstanding)
    if (!chain) {
        fetch(sb0);
        if (long_walk) chunked::chain_summaries<2>(table, pieces, seg * m - 1, seg * m, -1, sp, threadIdx.x);
        prepare(sb0, sh.step[0]);
        lds_barrier();
        if (sb0 + 1 < sb1) fetch(sb0 + 1);       // (not before the walk is over: its loads would wait behind these)
        if (seg > 0) lds_barrier();              // (the chained state has been read from where the next step's tables go)
        for (int sb = sb0; sb < sb1; sb++) {
            const int par = (sb - sb0) & 1;
            if (hf == 0 && y) {      // the masked matrix of block q
                const FwdTiles &sm = sh.step[par];
                const int row = 16 * q + n;
                f4 at = zero4(), a2 = zero4();
#pragma unroll
                for (int kk = 0; kk < 4; kk += 2) {
                    at = mma(along(sm.km, row, 16 * kk + 4 * g), along(sm.rm, row, 16 * kk + 4 * g), at);
                    a2 = mma(along(sm.km, row, 16 * kk + 16 + 4 * g), along(sm.rm, row, 16 * kk + 16 + 4 * g), a2);
                }
                const float rho = row_sum(sm.rho, row);
                at += a2;
#pragma unroll
                for (int e = 0; e < 4; e++) at[e] = 4 * g + e < n ? at[e] : 4 * g + e == n ? rho : 0.f;
                sh.at[par][q][lane] = at;
            }
            if (sb + 1 < sb1) {
                prepare(sb + 1, sh.step[par ^ 1]);
                fetch(min(sb + 2, sb1 - 1));
            }
            lds_barrier();
        }
        return;
    }
    // the state at the segment's start, put together while the other wavefronts prepare the first step:
    // S[kk][e] = S[key 16kk+4g+e][value 16q+n]
    f4 S[4];
    {
        if (seg > 0) {
            if (long_walk) chunked::chain_summaries<2>(table, pieces, seg * m - 1, seg * m, -1, sp, threadIdx.x);
            else chunked::chain_summaries<4>(table, pieces, seg * m - 1, seg * m, -1, sp, threadIdx.x);
            lds_barrier();
        }
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                S[kk][e] = seg > 0 ? table[(16 * kk + 4 * g + e) * LD + 16 * q + n] : sp[(16 * kk + 4 * g + e) * HEAD + 16 * q + n];
        lds_barrier();
        // Waited for here: left to the loop's first use of it, the wait would stand in the loop, and there it is one for the
        // stores of every step before (fp32 forward and backward of B8 T4096 H40, WKV5 1514 -> 1444 us, WKV6 1527 -> 1482).
#pragma unroll
        for (int kk = 0; kk < 4; kk++) asm volatile("" : "+v"(S[kk]));
    }
    const Out yo = out_of(y, (size_t)Tlen * C - h * HEAD);
    const uint32_t y_lane = (uint32_t)n * C + 16 * q + 4 * g;
    // a step token by token, from memory: the lane's sixteen keys of its value, added over the lane groups
    auto walk_tokens = [&](int sb) {
        const int t1 = min((sb + 1) * SB, Tlen);
#pragma unroll 1
        for (int t = sb * SB; t < t1; t++) {
            const size_t row = (size_t)t * C;
            const float vt = to_float(v[row + 16 * q + n]);
            float acc = 0.f, rho = 0.f;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                float r4[4], k4[4], w4[4], u4[4];
                const int key = 16 * kk + 4 * g;
                load4(r + row + key, r4); load4(k + row + key, k4); load4(wraw + (PER_TOKEN_W ? row : (size_t)h * HEAD) + key, w4); load4(u + h * HEAD + key, u4);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    rho = fmaf(r4[e] * u4[e], k4[e], rho);
                    acc = fmaf(r4[e], S[kk][e], acc);
                    S[kk][e] = fmaf(k4[e], vt, exp2_fast(log2_decay(w4[e], floor_decay)) * S[kk][e]);
                }
            }
            acc = over_groups(acc);
            rho = over_groups(rho);
            if (y && g == 0) put<T>(yo, t, C, 16 * q + n, fmaf(vt, rho, acc));
        }
    };
    int plain = any_plain(sh.step[0].plain);
    for (int sb = sb0; sb < sb1; sb++) {
        const int par = (sb - sb0) & 1;
        const FwdTiles &sm = sh.step[par];
        if (ckpt) {       // the state at the start of this step, 16 bytes per lane and tile
            f4 *cp = reinterpret_cast<f4 *>(ckpt + ((size_t)bh * (nsb + 1) + sb) * HEAD * HEAD) + q * 256 + lane;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) cp[64 * kk] = S[kk];
        }
        if (rarely(plain)) {
            walk_tokens(sb);
            lds_barrier();
            plain = any_plain(sh.step[par ^ 1].plain);
            continue;
        }
        f4 vv[4], yy[4];
#pragma unroll
        for (int blk = 0; blk < 4; blk++) {
            vv[blk] = across(sm.v, 16 * blk + 4 * g, 16 * q + n);
            f4 ya = zero4(), yb = zero4();
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                S[kk] *= *reinterpret_cast<const f4 *>(&sm.em[blk][16 * kk + 4 * g]);
                (kk & 1 ? yb : ya) = mma(S[kk], along(sm.rm, 16 * blk + n, 16 * kk + 4 * g), kk & 1 ? yb : ya);
                S[kk] = mma(across(sm.km, 16 * blk + 4 * g, 16 * kk + n), vv[blk], S[kk]);
                S[kk] *= *reinterpret_cast<const f4 *>(&sm.eb[blk][16 * kk + 4 * g]);
            }
            yy[blk] = ya + yb;
        }
        lds_barrier();
        plain = any_plain(sh.step[par ^ 1].plain);          // the next step's (read here, it costs the walk no wait)
        if (y) {
#pragma unroll
            for (int blk = 0; blk < 4; blk++)      // y^T: values 16q+4g .. +3 of token n
                put4<T>(yo, sb * SB + 16 * blk, C, y_lane, mma(vv[blk], sh.at[par][blk][lane], yy[blk]));
        }
    }
    if (seg == nseg - 1) {
        if (ckpt) {       // the final state takes the slot after the last step
            f4 *cp = reinterpret_cast<f4 *>(ckpt + ((size_t)bh * (nsb + 1) + nsb) * HEAD * HEAD) + q * 256 + lane;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) cp[64 * kk] = S[kk];
        }
        if (s_out) {
            float *op = s_out + (size_t)bh * HEAD * HEAD;
#pragma unroll
            for (int kk = 0; kk < 4; kk++)
#pragma unroll
                for (int e = 0; e < 4; e++) op[(16 * kk + 4 * g + e) * HEAD + 16 * q + n] = S[kk][e];
        }
    }
}

// ------------------------------------------------------------------------------------------------------ summary passes --
// What a piece of a segment does to a state handed in, or to a state gradient handed back (see summary_pass in
// wkv56_chunked.hip, whose walk away from the boundary and early stop this follows).  Four wavefronts: each prepares one
// block of a step and owns the values 16 w .. +15.
struct PassTiles {
    float a[SB * LD], b[SB * LD];        // forward: k e^{b-incl}, v;  backward: r e^{excl}, gy
    float dec[4][HEAD], tot[4][HEAD], fac[2][HEAD];
    int stop;
};
template <class T, class W, bool PER_TOKEN_W, bool BACKWARD>
__global__ __launch_bounds__(256) void summary_f32(int bh0, int Tlen, int C, int H, int nseg, int sps, int m, int pps,
        const T *__restrict__ a_in, const T *__restrict__ b_in, const W *__restrict__ wraw, float *__restrict__ part, int floor_decay)
{
    __shared__ __align__(16) PassTiles sm;
    const int units = (nseg - 1) * m;
    const int bh = bh0 + blockIdx.x / units, piece = (BACKWARD ? m : 0) + blockIdx.x % units, seg = piece / m, j = piece % m;
    const int b = bh / H, h = bh % H;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, n = lane & 15;
    {
        const size_t base = (size_t)b * Tlen * C + (size_t)h * HEAD;
        a_in += base; b_in += base;
        if (PER_TOKEN_W) wraw += base;
    }
    const int nsb = (Tlen + SB - 1) / SB;
    const int sb0 = seg * sps + j * pps, sb1 = min(min(nsb, (seg + 1) * sps), sb0 + pps), nsteps = sb1 - sb0;
    const float l_const = PER_TOKEN_W ? 0.f : log2_decay(to_float(wraw[h * HEAD + lane]), floor_decay);
    f4 X[4] = {zero4(), zero4(), zero4(), zero4()};       // X[kk][e] = X[key 16kk+4g+e][value 16wv+n]
    float R = 0.f;                                        // wavefront 0, lane = key
    T ta[16], tb[16];
    W tw[16];
    auto fetch = [&](int sb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = min(sb * SB + 16 * wv + i, Tlen - 1);
            ta[i] = *row_at(a_in, t, C, lane); tb[i] = *row_at(b_in, t, C, lane);
            if (PER_TOKEN_W) tw[i] = *row_at(wraw, t, C, lane);
        }
    };
    auto step_at = [&](int it) { return BACKWARD ? sb0 + it : sb1 - 1 - it; };
    if (nsteps > 0) fetch(step_at(0));
    if (tid < HEAD) sm.fac[0][tid] = 1.f;
    if (tid == 0) sm.stop = 0;
    bool stopped = false;
    for (int it = 0; it < nsteps; it++) {
        const int par = it & 1, sb = step_at(it);
        {
            float lw[16], run = 0.f;
#pragma unroll
            for (int i = 0; i < 16; i++)
                lw[i] = sb * SB + 16 * wv + i >= Tlen ? 0.f : PER_TOKEN_W ? log2_decay(to_float(tw[i]), floor_decay) : l_const;
#pragma unroll
            for (int x = 0; x < 16; x++) {                // backward: decay before the token; forward: decay after it
                const int i = BACKWARD ? x : 15 - x;
                const bool in = sb * SB + 16 * wv + i < Tlen;
                const int o = (16 * wv + i) * LD + lane;
                sm.a[o] = in ? to_float(ta[i]) * exp2_fast(run) : 0.f;
                sm.b[o] = in ? to_float(tb[i]) : 0.f;
                run += lw[i];
            }
            sm.tot[wv][lane] = run;
            sm.dec[wv][lane] = exp2_fast(run);
        }
        lds_barrier();
        if (it + 1 < nsteps) fetch(step_at(it + 1));
        if (wv == 0) {
            R += (sm.tot[0][lane] + sm.tot[1][lane]) + (sm.tot[2][lane] + sm.tot[3][lane]);
            sm.fac[par ^ 1][lane] = exp2_fast(R);
            if (__builtin_amdgcn_ballot_w64(R >= chunked::PASS_CUT_LOG2) == 0 && lane == 0) sm.stop = 1;
        }
        f4 Tt[4] = {zero4(), zero4(), zero4(), zero4()};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int blk = BACKWARD ? 3 - i : i;
            const f4 bb = across(sm.b, 16 * blk + 4 * g, 16 * wv + n);
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                if (i > 0) Tt[kk] *= *reinterpret_cast<const f4 *>(&sm.dec[blk][16 * kk + 4 * g]);
                Tt[kk] = mma(across(sm.a, 16 * blk + 4 * g, 16 * kk + n), bb, Tt[kk]);
            }
        }
#pragma unroll
        for (int kk = 0; kk < 4; kk++) X[kk] += Tt[kk] * *reinterpret_cast<const f4 *>(&sm.fac[par][16 * kk + 4 * g]);
        lds_barrier();
        if (sm.stop) { stopped = true; break; }
    }
    float *pp = part + ((size_t)bh * nseg * m + piece) * PART;
#pragma unroll
    for (int kk = 0; kk < 4; kk++)
#pragma unroll
        for (int e = 0; e < 4; e++) pp[(16 * kk + 4 * g + e) * HEAD + 16 * wv + n] = X[kk][e];
    if (wv == 0) pp[HEAD * HEAD + lane] = stopped ? 0.f : exp2_fast(R);
}

// ----------------------------------------------------------------------------------------------------------- backward --
// Eight wavefronts; the 64-token steps of a segment from the last to the first, in four parts between barriers:
//   prepare   wavefront (block q, half): eight tokens of one channel per lane
//   walk      wavefronts 0-3 (keys 16 w .. +15): the state forward from the step's checkpoint,  gy S1^T  of each block, then
//             the state gradient (value-major) backward,  v G1^T;  wavefronts 4-7: the masked matrices of one block each,
//             then the key-major gradient backward,  km G1  of the values 16 w .. +15
//   join      the masked matrices' products are added: d(rm), d(km) go to LDS, gv leaves
//   finish    wavefront (block q, half) again: gr, gk and the decay gradient of eight tokens of one channel per lane, in
//             whole rows
// Bound by the matrix pipe: 480 instructions of 32 clocks per SIMD and step, 432 of them in the walk, where a SIMD has one
// wavefront of either kind.  (With the matrices' products inside the walk, a barrier between the state's walk and the
// gradient's, and the key wavefronts finishing their own results: 28 k clocks a step against 15 k of matrix work.)
struct BwdTiles {
    float rm[SB * LD], km[SB * LD], v[SB * LD], gy[SB * LD], x[SB * LD], lw[SB * LD];
    float em[4][HEAD], eb[4][HEAD];
    f4 pm[4][64], pt[4][64], at[4][64];      // P (t > s): rows t, columns s;  P^T (s < t): rows s, columns t;  rm km^T (t >= s): rows t, columns s
    float dr[SB * LD], dk[SB * LD];          // d(rm), d(km)
    float rho[8][4][8], pdiag[SB], sums[8][HEAD];      // sums: of rm d(rm) - km d(km) over half a block
    alignas(16) int plain[8];                // half a block each: the step is walked token by token
};

template <class T, class W, bool PER_TOKEN_W>
__global__ __launch_bounds__(NT) void backward_f32(int bh0, int Tlen, int C, int H, int nseg, int sps, int m,
        const T *__restrict__ r, const T *__restrict__ k, const T *__restrict__ v, const W *__restrict__ wraw,
        const float *__restrict__ u, const T *__restrict__ gy, const float *__restrict__ gs_out, const float *__restrict__ ckpt,
        const float *__restrict__ gpart, T *__restrict__ gr, T *__restrict__ gk, T *__restrict__ gv, W *__restrict__ gw_tok,
        float *__restrict__ gw_part, float *__restrict__ gu_part, float *__restrict__ gs_in, int floor_decay)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    BwdTiles &sm = *reinterpret_cast<BwdTiles *>(smem_raw);
    const int bh = bh0 + blockIdx.x / nseg, seg = blockIdx.x % nseg, b = bh / H, h = bh % H;
    const int lane = threadIdx.x & 63, w8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, n = lane & 15;
    const bool keys = w8 < 4;
    const int q = w8 & 3, own = 16 * q + n;
    {
        const size_t base = (size_t)b * Tlen * C + (size_t)h * HEAD;
        r += base; k += base; v += base; gy += base; gr += base; gk += base; gv += base;
        if (PER_TOKEN_W) { wraw += base; gw_tok += base; }
    }
    const int nsb = (Tlen + SB - 1) / SB, sb0 = seg * sps, sb1 = min(nsb, (seg + 1) * sps);
    // the slot of a checkpoint that holds [key own][value 16kk+4g+e] (the forward's tiles are [key][value])
    const float *ck_lane = ckpt + (size_t)bh * (nsb + 1) * HEAD * HEAD + ((size_t)q * 64 + 16 * (n >> 2) + 4 * g) * 4 + (n & 3);

    // keys: G[kk][e] = G[key own][value 16kk+4g+e];  values: G[kk][e] = G[key 16kk+4g+e][value own]
    f4 G[4] = {zero4(), zero4(), zero4(), zero4()};
    float A = 0.f;                           // running sum of the decay gradient at the end of a step, key `lane`
    {
        float X[16];
        const float *ends = gs_out ? gs_out + (size_t)bh * HEAD * HEAD : nullptr;
        float *table = sm.dr;
        if (seg != nseg - 1) {
            chunked::chain_summaries<2>(table, gpart + (size_t)bh * nseg * m * PART, (seg + 1) * m, (nseg - 1 - seg) * m, 1, ends, threadIdx.x);
            lds_barrier();
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int x = 16 * (i >> 2) + 4 * g + (i & 3), key = keys ? own : x, value = keys ? x : own;
            X[i] = seg != nseg - 1 ? table[key * LD + value] : ends ? ends[key * HEAD + value] : 0.f;
        }
        if (keys) {       // anchored at the segment's end: sum_j G o S
            const float *cp = ck_lane + (size_t)sb1 * HEAD * HEAD;
#pragma unroll
            for (int i = 0; i < 16; i++) A = fmaf(X[i], cp[(i >> 2) * 1024 + (i & 3) * 4], A);
            A = chunked::group_sum4(A);
            if (g == 0) sm.sums[0][own] = A;
        }
#pragma unroll
        for (int i = 0; i < 16; i++) G[i >> 2][i & 3] = X[i];
    }
    float gu_acc = 0.f, gw_acc = 0.f;        // of the lane's tokens, key `lane`

    // preparing: block q, half hf, channel `lane`
    const int hf = w8 >> 2, tok0 = 16 * q + 8 * hf;
    const float uf = u[h * HEAD + lane];
    const float l_const = PER_TOKEN_W ? 0.f : log2_decay(to_float(wraw[h * HEAD + lane]), floor_decay);
    T tr[8], tk[8], tv[8], tg[8];
    W tw[8];
    auto fetch = [&](int sb, int lane) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int t = min(sb * SB + tok0 + i, Tlen - 1);
            tr[i] = *row_at(r, t, C, lane); tk[i] = *row_at(k, t, C, lane); tv[i] = *row_at(v, t, C, lane); tg[i] = *row_at(gy, t, C, lane);
            if (PER_TOKEN_W) tw[i] = *row_at(wraw, t, C, lane);
        }
    };
    auto prepare = [&](int sb, int lane) __attribute__((always_inline)) {
        float lw[8], x[8], p[8], m = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++)
            lw[i] = sb * SB + tok0 + i >= Tlen ? 0.f : PER_TOKEN_W ? log2_decay(to_float(tw[i]), floor_decay) : l_const;
        const float total = hf ? half_exponents<8, true>(lw, x) : half_exponents<8, false>(lw, x);
        (hf ? sm.eb : sm.em)[q][lane] = exp2_fast(total);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const bool in = sb * SB + tok0 + i < Tlen;
            const float rf = in ? to_float(tr[i]) : 0.f, kf = in ? to_float(tk[i]) : 0.f;
            const float vf = in ? to_float(tv[i]) : 0.f, gf = in ? to_float(tg[i]) : 0.f;
            const int o = (tok0 + i) * LD + lane;
            sm.rm[o] = rf * exp2_fast(x[i]);
            sm.km[o] = kf * exp2_fast(-(x[i] + lw[i]));
            sm.v[o] = vf;
            sm.gy[o] = gf;
            sm.x[o] = x[i];
            sm.lw[o] = lw[i];
            p[i] = rf * uf * kf;
            m = largest(m, rf, kf);
            m = largest(m, vf, gf);
            if (PER_TOKEN_W && (i & 1)) m = largest(m, lw[i - 1], lw[i]);          // (at most 8; for its NaN)
        }
        store_row_sums(p, sm.rho[2 * q + hf], lane);
        store_plain(&sm.plain[2 * q + hf], m, lane);
    };
    // For the walk token by token: r, k as they are, no exponents.  (Both kinds of wavefronts come here after work on the step
    // that is then done again, so that the flags are there by the time they are looked at; what others still read of
    // the tables meanwhile is of no use to them.)
    auto prepare_plain = [&](int sb, int lane) {
        fetch(sb, lane);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const bool in = sb * SB + tok0 + i < Tlen;
            const int o = (tok0 + i) * LD + lane;
            sm.rm[o] = in ? to_float(tr[i]) : 0.f;
            sm.km[o] = in ? to_float(tk[i]) : 0.f;
            sm.x[o] = 0.f;
        }
        fetch(max(sb - 1, sb0), lane);
        lds_barrier();
    };
    const size_t left = (size_t)Tlen * C - h * HEAD;
    const Out gro = out_of(gr, left), gko = out_of(gk, left), gwo = out_of(PER_TOKEN_W ? gw_tok : nullptr, PER_TOKEN_W ? left : 0);
    // dL/dlog w_t = A_t - km_t d(km)_t, A_t the running sum after token t.  plain: after a walk token by token, whose r, k, d(rm)
    // and d(km) carry no factor
    auto finish = [&](int sb, int lane, bool plain) __attribute__((always_inline)) {
        float rm[8], km[8], dr[8], dk[8], z[8], c[8], sum = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int o = (tok0 + i) * LD + lane;
            rm[i] = sm.rm[o]; km[i] = sm.km[o]; dr[i] = sm.dr[o]; dk[i] = sm.dk[o];
            z[i] = km[i] * dk[i];
            c[i] = fmaf(rm[i], dr[i], -z[i]);
            sum += c[i];
        }
        sm.sums[2 * q + hf][lane] = sum;
        lds_barrier();
        float run = A;
#pragma unroll
        for (int j = 7; j >= 0; j--) {
            const float x = sm.sums[j][lane];
            A += x;
            run += j > 2 * q + hf ? x : 0.f;
        }
#pragma unroll
        for (int i = 7; i >= 0; i--) {
            const int o = (tok0 + i) * LD + lane;
            const float x = sm.x[o], lw = sm.lw[o], ls = plain ? 0.f : lw, bonus = exp2_fast(ls) * sm.pdiag[tok0 + i], D = run - z[i];
            run += c[i];
            gu_acc = fmaf(rm[i] * km[i], bonus, gu_acc);
            const int t = sb * SB + tok0 + i;
            put<T>(gro, t, C, lane, exp2_fast(x) * fmaf(uf * km[i], bonus, dr[i]));
            put<T>(gko, t, C, lane, exp2_fast(-(x + ls)) * fmaf(uf * rm[i], bonus, dk[i]));
            if (PER_TOKEN_W) put<W>(gwo, t, C, lane, (floor_decay && lw <= LOG2_W_FLOOR) ? 0.f : D * (lw * LN2));
            else gw_acc += t < Tlen ? D : 0.f;
        }
    };
    // In the loops below a lane's indices come from an opaque copy of its number: addresses hoisted out of the loop would
    // live, and spill, across all of it.
#define WKV_F32_LANE                                                                      \
    int lane = lane0;                                                                     \
    asm volatile("" : "+v"(lane));                                                        \
    const int g = lane >> 4, n = lane & 15, own = 16 * q + n;
    const int lane0 = lane;
    lds_barrier();
    A = sm.sums[0][lane];
    lds_barrier();                                   // (before a step's sums go there)
    if (!keys) {
        const Out gvo = out_of(gv, left);
        fetch(sb1 - 1, lane);
        for (int sb = sb1 - 1; sb >= sb0; sb--) {
            WKV_F32_LANE
            prepare(sb, lane);
            lds_barrier();
            const int plain = any_plain(sm.plain);
            {       // the masked matrices of block q
                const int row = 16 * q + n;
                f4 p = zero4(), pT = zero4(), at = zero4();
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    const f4 a = along(sm.gy, row, 16 * kk + 4 * g), c = along(sm.v, row, 16 * kk + 4 * g);
                    p = mma(a, c, p);
                    pT = mma(c, a, pT);
                    at = mma(along(sm.rm, row, 16 * kk + 4 * g), along(sm.km, row, 16 * kk + 4 * g), at);
                }
                const float rho = row_sum(sm.rho, row);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int x = 4 * g + e;
                    if (x == n) sm.pdiag[row] = p[e];
                    p[e] = x > n ? p[e] : 0.f;
                    pT[e] = x < n ? pT[e] : 0.f;
                    at[e] = x > n ? at[e] : x == n ? rho : 0.f;
                }
                sm.pm[q][lane] = p; sm.pt[q][lane] = pT; sm.at[q][lane] = at;
            }
            fetch(max(sb - 1, sb0), lane);          // before this step's stores, see Out
            if (rarely(plain)) {
                prepare_plain(sb, lane);
#pragma unroll 1
                for (int i = SB - 1; i >= 0; i--) {
                    const float gt = sm.gy[i * LD + own];
                    float a = 0.f;
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) {
                        const f4 k4 = along(sm.km, i, 16 * kk + 4 * g), r4 = along(sm.rm, i, 16 * kk + 4 * g), l4 = along(sm.lw, i, 16 * kk + 4 * g);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            a = fmaf(k4[e], G[kk][e], a);
                            G[kk][e] = fmaf(r4[e], gt, exp2_fast(l4[e]) * G[kk][e]);
                        }
                    }
                    a = over_groups(a);
                    if (g == 0) put<T>(gvo, sb * SB + i, C, own, fmaf(row_sum(sm.rho, i), gt, a));
                }
                lds_barrier();
                lds_barrier();
                finish(sb, lane, true);
                lds_barrier();
                continue;
            }
            f4 gf[4], gvv[4];
#pragma unroll
            for (int blk = 3; blk >= 0; blk--) {
                gf[blk] = across(sm.gy, 16 * blk + 4 * g, own);
                f4 a = zero4(), c = zero4();
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    G[kk] *= *reinterpret_cast<const f4 *>(&sm.eb[blk][16 * kk + 4 * g]);
                    (kk & 1 ? c : a) = mma(G[kk], along(sm.km, 16 * blk + n, 16 * kk + 4 * g), kk & 1 ? c : a);
                    G[kk] = mma(across(sm.rm, 16 * blk + 4 * g, 16 * kk + n), gf[blk], G[kk]);
                    G[kk] *= *reinterpret_cast<const f4 *>(&sm.em[blk][16 * kk + 4 * g]);
                }
                gvv[blk] = a + c;
            }
            lds_barrier();
#pragma unroll
            for (int blk = 0; blk < 4; blk++)        // gv^T: values 16q+4g .. +3 of token n
                put4<T>(gvo, sb * SB + 16 * blk, C, (uint32_t)n * C + 16 * q + 4 * g, mma(gf[blk], sm.at[blk][lane], gvv[blk]));
            lds_barrier();
            finish(sb, lane, false);
            lds_barrier();
        }
    } else {
        f4 S[4];                                     // [key own][value 16kk+4g+e], from the step's checkpoint
        auto fetch_state = [&](int sb, int lane) __attribute__((always_inline)) {
            const int g = lane >> 4, n = lane & 15;
            const float *cp = ckpt + ((size_t)bh * (nsb + 1) + sb) * HEAD * HEAD + ((size_t)q * 64 + 16 * (n >> 2) + 4 * g) * 4 + (n & 3);
#pragma unroll
            for (int kk = 0; kk < 4; kk++)
#pragma unroll
                for (int e = 0; e < 4; e++) S[kk][e] = cp[kk * 1024 + e * 4];
        };
        fetch(sb1 - 1, lane);
        fetch_state(sb1 - 1, lane);
        for (int sb = sb1 - 1; sb >= sb0; sb--) {
            WKV_F32_LANE
            prepare(sb, lane);
            lds_barrier();
            const int plain = any_plain(sm.plain);
            f4 q1[4], q4[4];                         // rows: tokens of the block, column key own
#pragma unroll
            for (int blk = 0; blk < 4; blk++) {
                const float em = sm.em[blk][own];
                f4 a = zero4(), c = zero4();
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    S[kk] *= em;
                    (kk & 1 ? c : a) = mma(along(sm.gy, 16 * blk + n, 16 * kk + 4 * g), S[kk], kk & 1 ? c : a);
                }
                q1[blk] = a + c;
                if (blk < 3) {
                    const float eb = sm.eb[blk][own];
                    const f4 kf = across(sm.km, 16 * blk + 4 * g, own);
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) S[kk] = mma(across(sm.v, 16 * blk + 4 * g, 16 * kk + n), kf, S[kk]) * eb;
                }
            }
            if (rarely(plain)) {
                fetch_state(sb, lane);
                prepare_plain(sb, lane);
#pragma unroll 1
                for (int i = 0; i < SB; i++) {
                    const float kt = sm.km[i * LD + own], wt = exp2_fast(sm.lw[i * LD + own]);
                    float a = 0.f;
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) {
                        const f4 g4 = along(sm.gy, i, 16 * kk + 4 * g), v4 = along(sm.v, i, 16 * kk + 4 * g);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            a = fmaf(S[kk][e], g4[e], a);
                            S[kk][e] = fmaf(kt, v4[e], wt * S[kk][e]);
                        }
                    }
                    a = over_groups(a);
                    if (g == 0) sm.dr[i * LD + own] = a;
                }
                fetch_state(max(sb - 1, sb0), lane);
#pragma unroll 1
                for (int i = SB - 1; i >= 0; i--) {
                    const float rt = sm.rm[i * LD + own], wt = exp2_fast(sm.lw[i * LD + own]);
                    float a = 0.f;
#pragma unroll
                    for (int kk = 0; kk < 4; kk++) {
                        const f4 g4 = along(sm.gy, i, 16 * kk + 4 * g), v4 = along(sm.v, i, 16 * kk + 4 * g);
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            a = fmaf(G[kk][e], v4[e], a);
                            G[kk][e] = fmaf(rt, g4[e], wt * G[kk][e]);
                        }
                    }
                    a = over_groups(a);
                    if (g == 0) sm.dk[i * LD + own] = a;
                }
                lds_barrier();
                lds_barrier();
                finish(sb, lane, true);
                lds_barrier();
                continue;
            }
            fetch(max(sb - 1, sb0), lane);           // before this step's stores, see Out
            fetch_state(max(sb - 1, sb0), lane);
#pragma unroll
            for (int blk = 3; blk >= 0; blk--) {
                const float em = sm.em[blk][own], eb = sm.eb[blk][own];
                const f4 rf = across(sm.rm, 16 * blk + 4 * g, own);
                f4 a = zero4(), c = zero4();
#pragma unroll
                for (int kk = 0; kk < 4; kk++) {
                    G[kk] *= eb;
                    (kk & 1 ? c : a) = mma(along(sm.v, 16 * blk + n, 16 * kk + 4 * g), G[kk], kk & 1 ? c : a);
                    G[kk] = mma(across(sm.gy, 16 * blk + 4 * g, 16 * kk + n), rf, G[kk]) * em;
                }
                q4[blk] = a + c;
            }
            lds_barrier();
#pragma unroll
            for (int blk = 0; blk < 4; blk++) {
                const f4 dr = mma(sm.pt[blk][lane], across(sm.km, 16 * blk + 4 * g, own), q1[blk]);
                const f4 dk = mma(sm.pm[blk][lane], across(sm.rm, 16 * blk + 4 * g, own), q4[blk]);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int o = (16 * blk + 4 * g + e) * LD + own;
                    sm.dr[o] = dr[e];
                    sm.dk[o] = dk[e];
                }
            }
            lds_barrier();
            finish(sb, lane, false);
            lds_barrier();
        }
        if (gs_in && seg == 0) {
            float *gp = gs_in + (size_t)bh * HEAD * HEAD + own * HEAD;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) *reinterpret_cast<f4 *>(gp + 16 * kk + 4 * g) = G[kk];
        }
    }
#undef WKV_F32_LANE
    // sums over the segment's tokens: the eight wavefronts' shares in a fixed order
    float *red = sm.dr;
    red[w8 * HEAD + lane] = gu_acc;
    red[(8 + w8) * HEAD + lane] = gw_acc;
    lds_barrier();
    if (w8 == 0) {
        float su = 0.f, sw = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) { su += red[i * HEAD + lane]; sw += red[(8 + i) * HEAD + lane]; }
        const size_t po = ((size_t)(b * nseg + seg) * H + h) * HEAD + lane;
        gu_part[po] = su;
        if (!PER_TOKEN_W) {
            bool fl;
            const float l = log_decay(to_float(wraw[h * HEAD + lane]), floor_decay, &fl);
            gw_part[po] = fl ? 0.f : sw * l;
        }
    }
}

// ---------------------------------------------------------------------------------------------------------- launchers --
template <class T, class W, bool PT> struct Kernels {
    static constexpr auto *fwd = &forward_f32<T, W, PT>;
    static constexpr auto *bwd = &backward_f32<T, W, PT>;
    static hipError_t init() {
        hipError_t e = hipFuncSetAttribute((const void *)fwd, hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(FwdShared));
        if (e == hipSuccess) e = hipFuncSetAttribute((const void *)bwd, hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(BwdTiles));
        return e;
    }
    // ckpt, part as in chunked::forward_launch
    static hipError_t forward(hipStream_t s, int B, int Tlen, int C, int H, const void *r, const void *k, const void *v, const void *w,
                              const float *u, const float *s_in, void *y, float *s_out, float *ckpt, float *part,
                              const chunked::GroupPlan &plan, int floor_decay) {
        const int nsb = (Tlen + SB - 1) / SB, BH = B * H;
        const chunked::GroupPlan gp = part ? plan : chunked::GroupPlan{0, {1, nsb, 1, nsb}, {1, nsb, 1, nsb}};
        const chunked::SegPlan &pl = gp.b;
        const int nB = BH - gp.nA;
        if (pl.nseg > 1)
            hipLaunchKernelGGL((summary_f32<T, W, PT, false>), dim3(nB * (pl.nseg - 1) * pl.m), dim3(256), 0, s, gp.nA, Tlen, C, H, pl.nseg,
                               pl.sps, pl.m, pl.pps, (const T *)k, (const T *)v, (const W *)w, part, floor_decay);
        auto launch = [&](int bh0, int n, const chunked::SegPlan &x) {
            if (n > 0)
                hipLaunchKernelGGL((forward_f32<T, W, PT>), dim3(n * x.nseg), dim3(NT_FWD), sizeof(FwdShared), s, bh0, Tlen, C, H, x.nseg, x.sps,
                                   x.m, (const T *)r, (const T *)k, (const T *)v, (const W *)w, u, s_in, (T *)y, s_out, ckpt, part, floor_decay);
        };
        prof_begin(KID_CHUNK_FORWARD, s);
        launch(0, gp.nA, gp.a);
        launch(gp.nA, nB, pl);
        prof_end(KID_CHUNK_FORWARD, s);
        return hipGetLastError();
    }
    static hipError_t backward(hipStream_t s, int B, int Tlen, int C, int H, const void *r, const void *k, const void *v, const void *w,
                               const float *u, const float *s_in, const void *gy, const float *gs_out, void *gr, void *gk, void *gv, void *gw,
                               float *gu, float *gs_in, void *workspace, bool have_ckpt, int floor_decay) {
        const int BH = B * H;
        const chunked::GroupPlan gp = chunked::plan_groups(BH, Tlen, chunked::F32_COSTS);
        const chunked::Layout L = chunked::layout(B, Tlen, C, H, gp);
        const chunked::SegPlan &pl = gp.b;
        char *ws = (char *)workspace;
        float *ckpt = (float *)(ws + L.ckpt), *gpart = (float *)(ws + L.gpart);
        float *gu_one = (float *)(ws + L.sums), *gu_many = gu_one + (size_t)B * C;
        float *gw_one = gu_many + (size_t)B * pl.nseg * C, *gw_many = gw_one + (size_t)B * C;
        if (!have_ckpt) {
            hipError_t e = forward(s, B, Tlen, C, H, r, k, v, w, u, s_in, nullptr, nullptr, ckpt, pl.nseg > 1 ? (float *)(ws + L.part) : nullptr,
                                   gp, floor_decay);
            if (e != hipSuccess) return e;
        }
        const int nB = BH - gp.nA;
        if (pl.nseg > 1)
            hipLaunchKernelGGL((summary_f32<T, W, PT, true>), dim3(nB * (pl.nseg - 1) * pl.m), dim3(256), 0, s, gp.nA, Tlen, C, H, pl.nseg,
                               pl.sps, pl.m, pl.pps, (const T *)r, (const T *)gy, (const W *)w, gpart, floor_decay);
        auto launch = [&](int bh0, int n, const chunked::SegPlan &x, float *gw_part, float *gu_part) {
            if (n > 0)
                hipLaunchKernelGGL((backward_f32<T, W, PT>), dim3(n * x.nseg), dim3(NT), sizeof(BwdTiles), s, bh0, Tlen, C, H, x.nseg, x.sps, x.m,
                                   (const T *)r, (const T *)k, (const T *)v, (const W *)w, u, (const T *)gy, gs_out, ckpt, gpart, (T *)gr, (T *)gk,
                                   (T *)gv, PT ? (W *)gw : nullptr, gw_part, gu_part, gs_in, floor_decay);
        };
        prof_begin(KID_CHUNK_BACKWARD, s);
        launch(0, gp.nA, gp.a, gw_one, gu_one);
        launch(gp.nA, nB, pl, gw_many, gu_many);
        prof_end(KID_CHUNK_BACKWARD, s);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        return chunked::sum_partials_launch(s, B, C, H, gp.nA, pl.nseg, gu_one, gu_many, gu, PT ? nullptr : gw_one, gw_many, (float *)gw);
    }
};
// dtype, decay type and form of the decay -> the kernels for them
template <class F> static hipError_t with_kernels(int dtype, bool w16, bool per_token, F f) {
    if (!per_token) return dtype == 0 ? f(Kernels<float, float, false>()) : f(Kernels<f16, float, false>());
    if (dtype == 0) return f(Kernels<float, float, true>());
    return w16 ? f(Kernels<f16, f16, true>()) : f(Kernels<f16, float, true>());
}
static hipError_t init_kernels() {
    static PerDevice done;
    return done.once([] {
        hipError_t e = Kernels<float, float, false>::init();
        if (e == hipSuccess) e = Kernels<f16, float, false>::init();
        if (e == hipSuccess) e = Kernels<float, float, true>::init();
        if (e == hipSuccess) e = Kernels<f16, float, true>::init();
        if (e == hipSuccess) e = Kernels<f16, f16, true>::init();
        return e;
    });
}
// workspace as chunked::forward_launch's; keep: checkpoints at its start, else it holds the piece summaries alone.  State
// updated in place: the workgroups of later time segments would read what the last one's has overwritten, so the
// sequences run in one piece.
static hipError_t forward_launch(hipStream_t s, int dtype, bool per_token, bool w16, int B, int Tlen, int C, int H, const void *r, const void *k,
                                 const void *v, const void *w, const float *u, const float *s_in, void *y, float *s_out, void *workspace,
                                 bool keep, int floor_decay) {
    hipError_t e = init_kernels();
    if (e != hipSuccess) return e;
    const chunked::GroupPlan gp = chunked::plan_groups(B * H, Tlen, chunked::F32_COSTS);
    const chunked::Layout L = chunked::layout(B, Tlen, C, H, gp);
    char *ws = (char *)workspace;
    float *part = ws && gp.b.nseg > 1 && s_in != s_out ? (float *)(ws + (keep ? L.part : 0)) : nullptr;
    return with_kernels(dtype, w16, per_token, [&](auto kn) {
        return kn.forward(s, B, Tlen, C, H, r, k, v, w, u, s_in, y, s_out, ws && keep ? (float *)ws : nullptr, part, gp, floor_decay);
    });
}
static hipError_t backward_launch(hipStream_t s, int dtype, bool per_token, bool w16, int B, int Tlen, int C, int H, const void *r, const void *k,
                                  const void *v, const void *w, const float *u, const float *s_in, const void *gy, const float *gs_out, void *gr,
                                  void *gk, void *gv, void *gw, float *gu, float *gs_in, void *workspace, bool have_ckpt, int floor_decay) {
    hipError_t e = init_kernels();
    if (e != hipSuccess) return e;
    return with_kernels(dtype, w16, per_token, [&](auto kn) {
        return kn.backward(s, B, Tlen, C, H, r, k, v, w, u, s_in, gy, gs_out, gr, gk, gv, gw, gu, gs_in, workspace, have_ckpt, floor_decay);
    });
}

}  // namespace f32
}  // namespace wkv
