// RWKV-v4 WKV with (aa, bb, pp) state: one lane per (batch, channel) chain.
//
// The chain is serial in time, and a GPU holds few chains (B*C lanes), so two things set the speed: how many
// bytes each lane keeps in flight, and how many instructions the ONE wavefront that walks a chain has to issue per
// token.  For the first, blocks of 16 tokens of k, v (and gy) are fetched into registers several blocks ahead of the
// one being consumed; consecutive lanes are consecutive channels, so every load and store is a full coalesced row.
// For the second, only the recurrence itself stays with the walking wavefront; everything that can be formed from
// a block's starting state alone is handed to other wavefronts of the workgroup, which work on different blocks at
// the same time:
//   forward   wavefront 0 advances (p, q, o) and leaves the state at the start of every 16-token block in LDS;
//             wavefronts 1-3 take a block each (every third block) and form its 16 outputs from that state;
//   backward  wavefront 0 replays a block from the forward's checkpoint and leaves what the reverse walk needs of
//             its 16 tokens in LDS; wavefront 1 walks the block replayed just before backwards at the same time.
//             (More replaying wavefronts, the 16-byte fetches of the forward, or two pairs per workgroup were all
//             measured slower here: with the recurrence replayed the pass is bound by the instructions a compute
//             unit issues, not by one wavefront's.)
// Per token the arithmetic is kept short (one exponential per max-scaled pair, the bare reciprocal instruction) and
// free of branches, so that the tokens of a block are one straight-line stretch the scheduler can interleave.
//
// State convention (RWKV-v4neo/cuda/wkv_cuda_bf16.cu:30-52): (p, q, o) with
// p, q the decayed sums divided by e^{o}.  Backward carries the state gradient
// the same way, (gp, gq, go), and returns the decay gradient with respect to
// the raw time_decay parameter (:116-156).
//
// Backward never stores per-token intermediates for the whole sequence (the
// reference keeps three T-long arrays per lane): the forward sweep leaves a
// 5-float checkpoint (p, q, o, dp/dw, dq/dw) every 16 tokens, and the backward
// sweep replays one 16-token block at a time from its checkpoint.
#include "common.h"
#include <type_traits>

namespace wkv {

// one element of a result, stored with the non-temporal hint (results are not read again by these kernels)
__device__ __forceinline__ void stream1(float *p, float v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void stream1(bf16 *p, bf16 v) { __builtin_nontemporal_store(v.bits, &p->bits); }
__device__ __forceinline__ void stream1(f16 *p, f16 v) { __builtin_nontemporal_store(v.h, &p->h); }

constexpr int CK = 16;                 // tokens per checkpoint block
constexpr float NEG_HUGE = -1e38f;

struct Chain { float p, q, o, dp, dq; };

// Two terms scaled by a common maximum exponent, e^{a-m} and e^{b-m} with m = max(a, b): one of the two is
// exactly 1, so a pair costs one exponential, e^{-|a-b|}.
struct ExpPair { float first, second; bool first_is_max; };
__device__ __forceinline__ ExpPair exp_pair(float a, float b) {
    const float d = a - b, e = __expf(-fabsf(d));
    const bool fm = d >= 0.f;
    return ExpPair{fm ? 1.f : e, fm ? e : 1.f, fm};
}

// one token: output y and the pieces backward re-uses (1 / scaled denominator, the current token's scaled weight,
// the history's scaled weight, minus the scaling exponent); advances the chain
__device__ __forceinline__ float v4_step(Chain &s, float w, float u, float kk, float vv,
                                         float &iden, float &ec, float &hist_w, float &neg_m) {
    const float uk = u + kk;
    const ExpPair a = exp_pair(s.o, uk);
    hist_w = a.first;
    ec = a.second;
    neg_m = a.first_is_max ? -s.o : -uk;
    iden = __builtin_amdgcn_rcpf(hist_w * s.q + ec);      // the bare v_rcp_f32 (1 ulp), not a full division
    const float y = (hist_w * s.p + ec * vv) * iden;
    const float wo = w + s.o;
    const ExpPair d = exp_pair(wo, kk);
    const float dh = d.first, dc = d.second;
    s.dp = dh * (s.p + s.dp);
    s.dq = dh * (s.q + s.dq);
    s.p = fmaf(dh, s.p, dc * vv);
    s.q = fmaf(dh, s.q, dc);
    s.o = d.first_is_max ? wo : kk;
    return y;
}

// the recurrence alone: the same operations on (p, q, o, dp, dq) as v4_step, in the same order
__device__ __forceinline__ void v4_advance(Chain &s, float w, float kk, float vv) {
    const float wo = w + s.o;
    const ExpPair d = exp_pair(wo, kk);
    const float dh = d.first, dc = d.second;
    s.dp = dh * (s.p + s.dp);
    s.dq = dh * (s.q + s.dq);
    s.p = fmaf(dh, s.p, dc * vv);
    s.q = fmaf(dh, s.q, dc);
    s.o = d.first_is_max ? wo : kk;
}

// A block of 16 tokens x 64 chains of one tensor on its way from memory to the lanes that own the chains.  A
// wavefront can have 64 memory instructions in flight, so what it has in flight in bytes is set by the size of one:
//   WIDE   16 bytes per lane: lane l fetches W = 16 / sizeof(T) consecutive chains of token l / (64/W) of every
//          group of 64 / (64/W) tokens (a full 256- or 128-byte row segment per 64/W lanes); a block is 4 (fp32) or
//          2 (bf16, fp16) instructions.  The pieces reach their owners through LDS: written as they came,
//          [token][chain], read back one element per lane and token.  Needs C to be a multiple of W (a piece
//          never straddles two batch rows) and 16-byte aligned tensors.
//   narrow one element per lane and token: 16 instructions per block; any C.
// Either way the block ends up in the LDS area handed in as well as in the caller's registers.
template <class T, bool WIDE> struct V4In;
template <class T> struct V4In<T, false> {
    T val[CK];
    __device__ __forceinline__ void fetch(const T *p, int /*chain0*/, int idx, int /*BC*/, int C, int Tlen, int /*Tend*/, int t0, int /*lane*/) {
        const int b = idx / C, c = idx % C;
        const T *q = p + ((size_t)b * Tlen + t0) * C + c;
        if (t0 + CK <= Tlen) {          // whole block inside the sequence: no per-token checks
#pragma unroll
            for (int i = 0; i < CK; i++, q += C) val[i] = *q;
        } else {
#pragma unroll
            for (int i = 0; i < CK; i++, q += C) val[i] = t0 + i < Tlen ? *q : T{};
        }
    }
    __device__ __forceinline__ void spread(T *stage, int lane, T (&out)[CK]) const {
#pragma unroll
        for (int i = 0; i < CK; i++) { out[i] = val[i]; stage[i * 64 + lane] = val[i]; }
    }
};
template <class T> struct V4In<T, true> {
    static constexpr int W = 16 / sizeof(T), LPR = 64 / W, ROWS = 64 / LPR, NLD = CK / ROWS;
    typedef unsigned int piece_t __attribute__((ext_vector_type(4)));
    piece_t piece[NLD];
    // chain0: the wavefront's first chain (a multiple of 64); tokens from Tend on repeat the one before (never used)
    __device__ __forceinline__ void fetch(const T *p, int chain0, int /*idx*/, int BC, int C, int Tlen, int Tend, int t0, int lane) {
        const int q = min(chain0 + (lane % LPR) * W, BC - W);
        const T *row = p + (size_t)(q / C) * Tlen * C + q % C;
#pragma unroll
        for (int i = 0; i < NLD; i++)
            piece[i] = *reinterpret_cast<const piece_t *>(row + (size_t)min(t0 + i * ROWS + lane / LPR, Tend - 1) * C);
    }
    __device__ __forceinline__ void spread(T *stage, int lane, T (&out)[CK]) const {
#pragma unroll
        for (int i = 0; i < NLD; i++) *reinterpret_cast<piece_t *>(stage + (i * ROWS + lane / LPR) * 64 + (lane % LPR) * W) = piece[i];
#pragma unroll
        for (int i = 0; i < CK; i++) out[i] = stage[i * 64 + lane];
    }
};

// One token per sequence, nothing kept for a backward: one lane per chain, no staging (the general kernel brings eight
// wavefronts and up to 113 KB of LDS for 128 chains: B16 C2560 bf16 6.8 us on the GPU, and a call 12 us; with this kernel the
// host is what a call waits for, 6.7 us).  state_out may be state_in.
template <class T>
__global__ __launch_bounds__(256) void v4_decode(int BC, int C, const float *__restrict__ time_decay, const float *__restrict__ time_first,
        const T *__restrict__ k, const T *__restrict__ v, const float *s_in, T *__restrict__ y, float *s_out)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= BC) return;
    const int c = idx % C;
    Chain s{0.f, 0.f, NEG_HUGE, 0.f, 0.f};
    if (s_in) { s.p = s_in[idx * 3]; s.q = s_in[idx * 3 + 1]; s.o = s_in[idx * 3 + 2]; }
    float iden, ec, hw, nm;
    const float yy = v4_step(s, -__expf(time_decay[c]), time_first[c], to_float(k[idx]), to_float(v[idx]), iden, ec, hw, nm);
    y[idx] = from_float<T>(yy);
    if (s_out) { s_out[idx * 3] = s.p; s_out[idx * 3 + 1] = s.q; s_out[idx * 3 + 2] = s.o; }
}

// ---- Sequences cut in time.  A GPU full of chains has B*C / 64 wavefronts walking; with fewer the walk over T tokens is
// all there is to the time (some 50 ns a token forward, 125 backward, however few the chains).  Both recurrences are linear in
// their state, so a sequence may be cut into segments of whole blocks that run side by side (grid row = segment): a pass
// over all segments but one leaves what each adds to an empty state (its summary), and every segment starts by putting
// together the summaries before it (backward: after it).
struct Segment {
    int blk0, blk1;          // its blocks
    bool last;
    __device__ __forceinline__ Segment(int Tlen, int bps) {
        const int all = (Tlen + CK - 1) / CK;
        blk0 = blockIdx.y * bps;
        blk1 = min(blk0 + bps, all);
        last = blk1 == all;
    }
};
// a state after another L tokens whose summary is x: (p, q, o, dp, dq) of those tokens alone.  L steps without input take
// dp to e^{Lw} (dp + L p): every step adds p to dp before it decays both.
__device__ __forceinline__ void v4_append(Chain &s, float L, float w, const float (&x)[5]) {
    const float wo = fmaf(L, w, s.o);
    const ExpPair d = exp_pair(wo, x[2]);
    s.dp = fmaf(d.first, fmaf(L, s.p, s.dp), d.second * x[3]);
    s.dq = fmaf(d.first, fmaf(L, s.q, s.dq), d.second * x[4]);
    s.p = fmaf(d.first, s.p, d.second * x[0]);
    s.q = fmaf(d.first, s.q, d.second * x[1]);
    s.o = d.first_is_max ? wo : x[2];
}
// f(j, summary j) for n summaries from `first` in steps of `step`; four are in flight at a time.  part: [segment][N][B*C]
template <int N, class F>
__device__ __forceinline__ void for_summaries(const float *part, int BC, int idx, int first, int n, int step, F f) {
    for (int i = 0; i < n; i += 4) {
        float x[4][N];
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int e = 0; e < N; e++) x[a][e] = part[((size_t)(first + step * min(i + a, n - 1)) * N + e) * BC + idx];
#pragma unroll
        for (int a = 0; a < 4; a++)
            if (i + a < n) f(first + step * (i + a), x[a]);
    }
}
// The two summary passes: one wavefront per 64 chains and segment, SW segments per workgroup, the inputs of SD blocks in
// registers.  Forward: (p, q, o, dp, dq) of segments 0 .. nseg - 2.
constexpr int SW = 4, SD = 2;
template <class T>
__global__ __launch_bounds__(64 * SW) void v4_summary_forward(int BC, int Tlen, int C, const float *__restrict__ time_decay,
        const T *__restrict__ k, const T *__restrict__ v, float *__restrict__ part, int nseg, int bps)
{
    const int lane = threadIdx.x & 63, seg = __builtin_amdgcn_readfirstlane(blockIdx.y * SW + (threadIdx.x >> 6));
    const int idx = blockIdx.x * 64 + lane;
    if (seg >= nseg - 1 || idx >= BC) return;
    const float w = -__expf(time_decay[idx % C]);
    V4In<T, false> ik[SD], iv[SD];          // (every block of these segments is a whole one)
    const int blk0 = seg * bps, blk1 = blk0 + bps;
    auto fetch = [&](int blk, V4In<T, false> &a, V4In<T, false> &b) __attribute__((always_inline)) {
        const int t0 = min(blk, blk1 - 1) * CK;          // (past the end the last block again, unused)
        a.fetch(k, 0, idx, BC, C, Tlen, Tlen, t0, lane);
        b.fetch(v, 0, idx, BC, C, Tlen, Tlen, t0, lane);
    };
#pragma unroll
    for (int d = 0; d < SD; d++) fetch(blk0 + d, ik[d], iv[d]);
    Chain s{0.f, 0.f, NEG_HUGE, 0.f, 0.f};
    for (int blk = blk0; blk < blk1; blk += SD)
#pragma unroll
        for (int d = 0; d < SD; d++) {
            if (blk + d >= blk1) break;
#pragma unroll
            for (int i = 0; i < CK; i++) v4_advance(s, w, to_float(ik[d].val[i]), to_float(iv[d].val[i]));
            if (blk + d + SD < blk1) fetch(blk + d + SD, ik[d], iv[d]);
        }
    float *o = part + (size_t)seg * 5 * BC + idx;
    o[0] = s.p; o[BC] = s.q; o[2 * (size_t)BC] = s.o; o[3 * (size_t)BC] = s.dp; o[4 * (size_t)BC] = s.dq;
}
// Backward: what the state gradient at the start of segments 1 .. nseg - 1 holds of their own tokens.  A token's share
// decays over the tokens before it, so with the exponent counted from the segment's start the sum can be taken in the order of
// the replay, and no second walk is needed.
template <class T>
__global__ __launch_bounds__(64 * SW) void v4_summary_backward(int BC, int Tlen, int C, const float *__restrict__ time_decay,
        const float *__restrict__ time_first, const T *__restrict__ k, const T *__restrict__ v, const T *__restrict__ gy,
        const float *__restrict__ ckpt, float *__restrict__ part, int nseg, int bps)
{
    const int lane = threadIdx.x & 63, seg = __builtin_amdgcn_readfirstlane(1 + blockIdx.y * SW + (threadIdx.x >> 6));
    const int idx = blockIdx.x * 64 + lane;
    if (seg >= nseg || idx >= BC) return;
    // (bounded: from time_decay = 89 on the decay is e^-inf, and no token before the segment's first, 0 times that, is not a number)
    const float w = fmaxf(-__expf(time_decay[idx % C]), -1e30f), u = time_first[idx % C];
    V4In<T, false> ik[SD], iv[SD], ig[SD];
    const int blk0 = seg * bps, blk1 = min(blk0 + bps, (Tlen + CK - 1) / CK);
    auto fetch = [&](int blk, int d) __attribute__((always_inline)) {
        const int t0 = min(blk, blk1 - 1) * CK;
        ik[d].fetch(k, 0, idx, BC, C, Tlen, Tlen, t0, lane);
        iv[d].fetch(v, 0, idx, BC, C, Tlen, Tlen, t0, lane);
        ig[d].fetch(gy, 0, idx, BC, C, Tlen, Tlen, t0, lane);
    };
#pragma unroll
    for (int d = 0; d < SD; d++) fetch(blk0 + d, d);
    const float *cp = ckpt + (size_t)blk0 * 5 * BC + idx;
    Chain s{cp[0], cp[BC], cp[2 * (size_t)BC], 0.f, 0.f};
    float gp = 0.f, gq = 0.f, go = NEG_HUGE;
    for (int blk = blk0; blk < blk1; blk += SD)
#pragma unroll
        for (int d = 0; d < SD; d++) {
            if (blk + d >= blk1) break;
            const int cnt = min(CK, Tlen - (blk + d) * CK);
            const float before = (float)((blk + d - blk0) * CK);
#pragma unroll
            for (int i = 0; i < CK; i++) {
                if (i < cnt) {
                    float iden, ec, hw, nm;
                    const float ys = v4_step(s, w, u, to_float(ik[d].val[i]), to_float(iv[d].val[i]), iden, ec, hw, nm);
                    const float at = fmaf(before + i, w, nm);
                    const ExpPair e = exp_pair(go, at);
                    const float add = to_float(ig[d].val[i]) * iden * e.second;
                    gp = fmaf(e.first, gp, add);
                    gq = fmaf(e.first, gq, -add * ys);
                    go = e.first_is_max ? go : at;
                }
            }
            if (blk + d + SD < blk1) fetch(blk + d + SD, d);
        }
    float *o = part + (size_t)seg * 3 * BC + idx;
    o[0] = gp; o[BC] = gq; o[2 * (size_t)BC] = go;
}

// Forward.  y == nullptr: only checkpoints / final state are produced.
// ckpt layout: [block][5][B*C].
// Four wavefronts per 64 chains.  One walks the chain, V4_YW blocks (a lap) between two workgroup barriers, and
// leaves in LDS the state at the start of each block and the block's k and v; each of the other three forms the
// outputs of one block of the lap before from what it finds there (it reads nothing from memory).  The walking
// wavefront's inputs wait in registers as they came, two laps deep (converting at the fetch would make every load
// wait for its data on the spot, and nothing would be in flight); register sets and LDS slots are fixed per use, two
// laps written out.
constexpr int V4_YW = 3, V4_GROUPS = 2;
template <class T, bool WIDE>
__global__ __launch_bounds__(64 * (1 + V4_YW) * V4_GROUPS) void v4_forward(int BC, int Tlen, int C, const float *__restrict__ time_decay,
        const float *__restrict__ time_first, const T *__restrict__ k, const T *__restrict__ v,
        const float *__restrict__ s_in, T *__restrict__ y, float *__restrict__ s_out, float *__restrict__ ckpt,
        const float *__restrict__ part, int bps)
{
    __shared__ float start_all[V4_GROUPS][2 * V4_YW][5][64];      // the state at a block's start: p, q, o (and dp, dq for the checkpoint)
    // k and v of the blocks of two laps, [token][chain]: left there by the walking wavefront on its way (it is also
    // how the 16-byte pieces reach their owners), read by the wavefront that forms the block's outputs a lap later
    extern __shared__ __align__(16) unsigned char kv_raw[];          // v4_forward_lds<T>() bytes
    typedef T KvBlock[CK * 64];
    KvBlock (*kv_all)[2 * V4_YW][2] = reinterpret_cast<KvBlock (*)[2 * V4_YW][2]>(kv_raw);
    // A workgroup is two groups of four wavefronts, 64 chains each.  The walking wavefront is the first of its four in
    // group 0 and the second in group 1: wavefronts go to the four SIMDs in turn, and two walkers on one SIMD would
    // share the one resource they are short of.
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), grp = wave >> 2, wl = wave & 3;
    const int role = wl == grp ? 0 : (wl < grp ? wl + 1 : wl);       // 0: walks the chain; 1 + r: outputs of every third block
    // (lanes and groups past the last chain stay, the 16-byte fetches being a wavefront's joint work and the barriers
    // the workgroup's: they read the last chains' inputs and write nothing)
    const int chain_grp = (blockIdx.x * V4_GROUPS + grp) * 64, chain0 = min(chain_grp, (BC - 1) / 64 * 64);
    const int idx = min(chain0 + lane, BC - 1);
    const bool live = chain_grp + lane < BC;
    float (*start)[5][64] = start_all[grp];
    const int b = idx / C, c = idx % C;
    const float w = -__expf(time_decay[c]), u = time_first[c];
    const size_t base = (size_t)b * Tlen * C + c;
    const Segment sg(Tlen, bps);
    const int blk0 = sg.blk0, nblk = sg.blk1, nlap = (nblk - blk0 + V4_YW - 1) / V4_YW;          // (nblk: the segment's end)
    const int Tend = min(Tlen, nblk * CK);
    typedef V4In<T, WIDE> In;

    if (role == 0) {
        Chain s{0.f, 0.f, NEG_HUGE, 0.f, 0.f};
        if (s_in) { s.p = s_in[idx * 3]; s.q = s_in[idx * 3 + 1]; s.o = s_in[idx * 3 + 2]; }
        // two laps of blocks: one being consumed, one in flight (named, not an array: every use is a fixed register set)
        static_assert(V4_YW == 3, "the laps are written out for three blocks");
        In k0, k1, k2, k3, k4, k5, v0, v1, v2, v3, v4, v5;
        // (The 16-byte fetches of the two-byte types are unconditional, also for blocks past the end, where they
        // repeat the last token and nobody uses them: after a load inside a branch the compiler waits for everything
        // outstanding instead of for the block it needs.  Measured at B8 T4096 C4096: bf16 forward 265 -> 259 us; fp32,
        // whose laps in flight are twice the bytes, 316 -> 331 us, so it keeps the conditional fetches.)
        constexpr bool AHEAD = WIDE && sizeof(T) == 2;
        auto first = [&](int d, In &ik, In &iv) __attribute__((always_inline)) {
            const int t0 = (blk0 + d) * CK;
            if (AHEAD || blk0 + d < nblk) { ik.fetch(k, chain0, idx, BC, C, Tlen, Tend, t0, lane); iv.fetch(v, chain0, idx, BC, C, Tlen, Tend, t0, lane); }
        };
        first(0, k0, v0); first(1, k1, v1); first(2, k2, v2); first(3, k3, v3); first(4, k4, v4); first(5, k5, v5);
        for_summaries<5>(part, BC, idx, 0, blk0 / bps, 1, [&](int, const float (&x)[5]) __attribute__((always_inline)) {
            v4_append(s, (float)(bps * CK), w, x);
        });
        auto block = [&](int blk, int slot, In &ik, In &iv) __attribute__((always_inline)) {
            if (!AHEAD && blk >= nblk) return;
            const bool on = blk < nblk;          // scalar
            T kk[CK], vv[CK];
            if (on) {
            // (the block's checkpoint is written by the wavefront that forms its outputs, from these five values: this
            // wavefront then has loads outstanding and nothing else, and loads alone are counted in order, so that a wait
            // for one block's inputs does not wait for the blocks fetched after it; with a store among them it would)
            start[slot][0][lane] = s.p; start[slot][1][lane] = s.q; start[slot][2][lane] = s.o;
            start[slot][3][lane] = s.dp; start[slot][4][lane] = s.dq;
            ik.spread(kv_all[grp][slot][0], lane, kk);
            iv.spread(kv_all[grp][slot][1], lane, vv);
            }
            const int nb = blk + 2 * V4_YW;
            if (AHEAD || nb < nblk) { ik.fetch(k, chain0, idx, BC, C, Tlen, Tend, nb * CK, lane); iv.fetch(v, chain0, idx, BC, C, Tlen, Tend, nb * CK, lane); }
            if (!on) return;
            const int t0 = blk * CK, cnt = min(CK, Tlen - t0);
            if (cnt == CK) {
#pragma unroll
                for (int i = 0; i < CK; i++) v4_advance(s, w, to_float(kk[i]), to_float(vv[i]));
            } else {
#pragma unroll
                for (int i = 0; i < CK; i++)
                    if (i < cnt) v4_advance(s, w, to_float(kk[i]), to_float(vv[i]));
            }
        };
        for (int rd = 0; rd <= nlap; rd += 2) {
            const int b0 = blk0 + rd * V4_YW;
            block(b0, 0, k0, v0); block(b0 + 1, 1, k1, v1); block(b0 + 2, 2, k2, v2);
            lds_barrier();
            block(b0 + 3, 3, k3, v3); block(b0 + 4, 4, k4, v4); block(b0 + 5, 5, k5, v5);
            lds_barrier();                       // (both halves always: blocks past the end do nothing)
        }
        if (s_out && live && sg.last) { s_out[idx * 3] = s.p; s_out[idx * 3 + 1] = s.q; s_out[idx * 3 + 2] = s.o; }
    } else {
        const int r = role - 1;
        // the outputs of this wavefront's block of lap pr (whose starting state and inputs wait in slot `slot`)
        auto outputs = [&](int pr, int slot) __attribute__((always_inline)) {
            const int blk = blk0 + pr * V4_YW + r;
            if (pr < 0 || blk >= nblk) return;
            if (ckpt && live) {
                float *cp = ckpt + (size_t)blk * 5 * BC + idx;
                cp[0] = start[slot][0][lane]; cp[BC] = start[slot][1][lane]; cp[2 * (size_t)BC] = start[slot][2][lane];
                cp[3 * (size_t)BC] = start[slot][3][lane]; cp[4 * (size_t)BC] = start[slot][4][lane];
            }
            if (!y) return;
            Chain s{start[slot][0][lane], start[slot][1][lane], start[slot][2][lane], 0.f, 0.f};
            const T *ks = kv_all[grp][slot][0], *vs = kv_all[grp][slot][1];
            T kk[CK], vv[CK];
#pragma unroll
            for (int i = 0; i < CK; i++) { kk[i] = ks[i * 64 + lane]; vv[i] = vs[i * 64 + lane]; }
            const int t0 = blk * CK, cnt = min(CK, Tlen - t0);
            T *yp = y + base + (size_t)t0 * C;
            if (cnt == CK) {
#pragma unroll
                for (int i = 0; i < CK; i++, yp += C) {
                    float iden, ec, hw, nm;
                    const float yy = v4_step(s, w, u, to_float(kk[i]), to_float(vv[i]), iden, ec, hw, nm);
                    if (live) stream1(yp, from_float<T>(yy));
                }
            } else {
#pragma unroll
                for (int i = 0; i < CK; i++, yp += C)
                    if (i < cnt) {
                        float iden, ec, hw, nm;
                        const float yy = v4_step(s, w, u, to_float(kk[i]), to_float(vv[i]), iden, ec, hw, nm);
                        if (live) stream1(yp, from_float<T>(yy));
                    }
            }
        };
        for (int rd = 0; rd <= nlap; rd += 2) {       // in lap rd: the block of lap rd-1
            outputs(rd - 1, V4_YW + r);
            lds_barrier();
            outputs(rd, r);
            lds_barrier();
        }
    }
}

// Backward: two wavefronts per 64 chains.  Replaying a block from its checkpoint does not depend on the reverse
// walk of the blocks after it, so the two halves of the work run side by side: wavefront 0 replays block b (and
// sums the decay / bonus gradients), leaving y, 1/denominator, the current token's weight and the scaling exponent
// of its 16 tokens in LDS; wavefront 1 meanwhile walks block b+1 backwards from what wavefront 0 left the step
// before.  One workgroup barrier per block; RB LDS buffers and RB register sets of inputs (one being consumed,
// the others in flight) used in turn.
constexpr int RB = 4;
struct V4Replay { float ys[CK][64], iden[CK][64], ec[CK][64], neg_m[CK][64]; };

// CUT: for sequences cut in time.  bf16 and fp16 sequences in one piece have a kernel of their own, because with the segment's bounds in
// registers and the summaries' loop in it the compiler schedules the walk worse: bf16 B8 T4096 C4096 621 us without them, 711 with
// (fp32 gains nothing: 665 and 661).
template <class T, bool CUT>
__global__ __launch_bounds__(128) void v4_backward(int BC, int Tlen, int C, const float *__restrict__ time_decay,
        const float *__restrict__ time_first, const T *__restrict__ k, const T *__restrict__ v,
        const T *__restrict__ gy, const float *__restrict__ gs_out, const float *__restrict__ ckpt,
        float *__restrict__ gw_part, float *__restrict__ gu_part, T *__restrict__ gk, T *__restrict__ gv,
        float *__restrict__ gs_in, const float *__restrict__ part, int bps)
{
    __shared__ V4Replay sh[RB];
    const int lane = threadIdx.x & 63, role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int idx = blockIdx.x * 64 + lane;
    if (idx >= BC) return;          // (the same lanes leave in both wavefronts; the barriers count wavefronts)
    const int b = idx / C, c = idx % C;
    const float w = -__expf(time_decay[c]), u = time_first[c];
    const size_t base = (size_t)b * Tlen * C + c;
    const int all = (Tlen + CK - 1) / CK, blk0 = CUT ? blockIdx.y * bps : 0, end = CUT ? min(blk0 + bps, all) : all;
    const int nblk = CUT ? end - blk0 : all;          // the segment's
    const bool last = !CUT || end == all;

    // RB blocks of k, v, gy per lane: one being consumed, the others in flight
    T bk[RB][CK], bv[RB][CK], bg[RB][CK];        // (as they came; converted where they are used)
    auto fetch = [&](int blk, T (&kk)[CK], T (&vv)[CK], T (&gg)[CK]) {
        const int t0 = blk * CK;
        const size_t o0 = base + (size_t)t0 * C;
        const T *kp = k + o0, *vp = v + o0, *gp_ = gy + o0;
        if (t0 + CK <= Tlen) {          // whole block inside the sequence: no per-token checks
#pragma unroll
            for (int i = 0; i < CK; i++, kp += C, vp += C, gp_ += C) { kk[i] = *kp; vv[i] = *vp; gg[i] = *gp_; }
        } else {
#pragma unroll
            for (int i = 0; i < CK; i++, kp += C, vp += C, gp_ += C) {
                const bool in = t0 + i < Tlen;
                kk[i] = in ? *kp : T{};
                vv[i] = in ? *vp : T{};
                gg[i] = in ? *gp_ : T{};
            }
        }
    };
    auto load_ckpt = [&](int blk) {
        const float *cp = ckpt + (size_t)blk * 5 * BC + idx;
        return Chain{cp[0], cp[BC], cp[2 * (size_t)BC], cp[3 * (size_t)BC], cp[4 * (size_t)BC]};
    };

    if (role == 0) {
        // ---------------- replay: step j handles block end-1-j, register set and LDS buffer j % RB
        float acc_w = 0.f, acc_u = 0.f;
        Chain bs[RB];
#pragma unroll
        for (int d = 0; d < RB; d++)
            if (nblk - 1 - d >= 0) { fetch(end - 1 - d, bk[d], bv[d], bg[d]); bs[d] = load_ckpt(end - 1 - d); }
        auto replay = [&](auto full_tag, int blk, T (&kk)[CK], T (&vv)[CK], T (&gg)[CK], Chain s, V4Replay &out) {
            constexpr bool FULL = decltype(full_tag)::value;
            const int cnt = FULL ? CK : Tlen - blk * CK;
#pragma unroll
            for (int i = 0; i < CK; i++) {
                if (FULL || i < cnt) {
                    const float dp0 = s.dp, dq0 = s.dq;
                    float hw, iden, ec, nm;
                    const float ki = to_float(kk[i]), vi = to_float(vv[i]), gi = to_float(gg[i]);
                    const float yy = v4_step(s, w, u, ki, vi, iden, ec, hw, nm);
                    acc_w += gi * (dp0 - dq0 * yy) * iden * hw;
                    acc_u += gi * (vi - yy) * ec * iden;
                    out.ys[i][lane] = yy; out.iden[i][lane] = iden; out.ec[i][lane] = ec; out.neg_m[i][lane] = nm;
                }
            }
            if (last && blk == end - 1 && gs_out) {       // gradient arriving through the state handed out
                const float gp = gs_out[idx * 3], gq = gs_out[idx * 3 + 1];
                const float go = (gp == 0.f && gq == 0.f) ? NEG_HUGE : gs_out[idx * 3 + 2];
                acc_w += (gp * s.dp + gq * s.dq) * __expf(s.o + go);
            }
        };
        auto step = [&](int j, T (&kk)[CK], T (&vv)[CK], T (&gg)[CK], Chain &cs, V4Replay &out) {
            const int blk = end - 1 - j;
            if (blk >= blk0) {
                if ((blk + 1) * CK <= Tlen) replay(std::true_type{}, blk, kk, vv, gg, cs, out);
                else replay(std::false_type{}, blk, kk, vv, gg, cs, out);
                if (blk - RB >= blk0) { fetch(blk - RB, kk, vv, gg); cs = load_ckpt(blk - RB); }
            }
            lds_barrier();
        };
        for (int j = 0; j <= nblk; j += RB) {
#pragma unroll
            for (int d = 0; d < RB; d++)
                if (j + d <= nblk) step(j + d, bk[d], bv[d], bg[d], bs[d], sh[d]);
        }
        const size_t o = (CUT ? (size_t)blockIdx.y * BC : 0) + idx;
        gw_part[o] = acc_w * w;
        gu_part[o] = acc_u;
    } else {
        // ---------------- reverse walk: step j handles block end-j (none at j = 0), register set and buffer (j-1) % RB
        float gp = 0.f, gq = 0.f, go = NEG_HUGE;
        if (gs_out) {
            gp = gs_out[idx * 3]; gq = gs_out[idx * 3 + 1]; go = gs_out[idx * 3 + 2];
            if (gp == 0.f && gq == 0.f) go = NEG_HUGE;
        }
#pragma unroll
        for (int d = 0; d < RB; d++)
            if (nblk - 1 - d >= 0) fetch(end - 1 - d, bk[d], bv[d], bg[d]);
        if (!last) {          // the segments after this one, from the last
            const int nseg = gridDim.y, seg = blockIdx.y, tail = Tlen - (nseg - 1) * bps * CK;          // tokens of the last
            for_summaries<3>(part, BC, idx, nseg - 1, nseg - 1 - seg, -1, [&](int j, const float (&x)[3]) __attribute__((always_inline)) {
                const float wg = fmaf((float)(j == nseg - 1 ? tail : bps * CK), w, go);
                const ExpPair e = exp_pair(wg, x[2]);
                gp = fmaf(e.first, gp, e.second * x[0]);
                gq = fmaf(e.first, gq, e.second * x[1]);
                go = e.first_is_max ? wg : x[2];
            });
        }
        auto walk = [&](auto full_tag, int blk, T (&kk)[CK], T (&vv)[CK], T (&gg)[CK], const V4Replay &in) {
            constexpr bool FULL = decltype(full_tag)::value;
            const int t0 = blk * CK, cnt = FULL ? CK : Tlen - t0;
            const size_t oe = base + (size_t)(t0 + CK - 1) * C;
            T *gkp = gk + oe, *gvp = gv + oe;
#pragma unroll
            for (int i = CK - 1; i >= 0; i--, gkp -= C, gvp -= C) {
                if (FULL || i < cnt) {
                    const float ys = in.ys[i][lane], iden = in.iden[i][lane], ec = in.ec[i][lane], nm = in.neg_m[i][lane];
                    const float ki = to_float(kk[i]), vi = to_float(vv[i]), gi = to_float(gg[i]);
                    const float direct = gi * iden * ec;
                    const float later = __expf(ki + go);
                    stream1(gkp, from_float<T>(direct * (vi - ys) + later * (gp * vi + gq)));
                    stream1(gvp, from_float<T>(direct + later * gp));
                    const float wg = w + go;
                    const ExpPair e = exp_pair(wg, nm);      // gy_t / den_t carries the exponent -m_t
                    const float add = gi * iden * e.second;
                    gp = fmaf(e.first, gp, add);
                    gq = fmaf(e.first, gq, -add * ys);
                    go = e.first_is_max ? wg : nm;
                }
            }
        };
        auto step = [&](int j, T (&kk)[CK], T (&vv)[CK], T (&gg)[CK], const V4Replay &in) {
            const int blk = end - j;
            if (j >= 1) {
                if ((blk + 1) * CK <= Tlen) walk(std::true_type{}, blk, kk, vv, gg, in);
                else walk(std::false_type{}, blk, kk, vv, gg, in);
                if (blk - RB >= blk0) fetch(blk - RB, kk, vv, gg);
            }
            lds_barrier();
        };
        for (int j = 0; j <= nblk; j += RB) {
#pragma unroll
            for (int d = 0; d < RB; d++) {
                constexpr int dummy = 0; (void)dummy;
                const int e = (d + RB - 1) % RB;
                if (j + d <= nblk) step(j + d, bk[e], bv[e], bg[e], sh[e]);
            }
        }
        if (gs_in && blk0 == 0) { gs_in[idx * 3] = gp; gs_in[idx * 3 + 1] = gq; gs_in[idx * 3 + 2] = go; }
    }
}

// g_time_decay and g_time_first: the rows of the partial sums, one per batch row and segment, in a fixed order: 32 columns x 8
// row groups per workgroup, grid row 0 the first, 1 the second
__global__ __launch_bounds__(256) void v4_sum(int rows, int C, const float *__restrict__ gw_part, const float *__restrict__ gu_part,
                                              float *__restrict__ gtd, float *__restrict__ gtf) {
    __shared__ float red[8][32];
    const float *in = blockIdx.y ? gu_part : gw_part;
    const int lane = threadIdx.x & 31, rg = threadIdx.x >> 5, c = blockIdx.x * 32 + lane;
    float s = 0.f;
    if (c < C) {
#pragma unroll 4
        for (int r = rg; r < rows; r += 8) s += in[(size_t)r * C + c];
    }
    red[rg][lane] = s;
    __syncthreads();
    if (rg != 0 || c >= C) return;
#pragma unroll
    for (int g = 1; g < 8; g++) s += red[g][lane];
    (blockIdx.y ? gtf : gtd)[c] = s;
}

static bool overlap(const float *a, const float *b, size_t bytes) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return a && b && x < y + bytes && y < x + bytes;
}

// Segments and blocks per segment.  As many segments as give every compute unit two wavefronts to walk with, or four where
// that leaves fewer than eight; at least two blocks each.  The passes over the summaries read the inputs once more, so a
// sequence is cut only where its chains take less than two thirds of the compute units (six segments or more) and where it has 16 blocks.
// Measured, fp32 forward+backward of whole calls in us, one piece against the rule's: 12 wavefronts of chains (B1 C768), T 4096
// 731 -> 80, T 1000 188 -> 52, T 256 58 -> 56 (T 128 48 -> 55: not cut); 40 (B1 C2560), T 4096 733 -> 173; 128 (B2 C4096) 802 ->
// 424; 160 (B4 C2560), T 1024 200 -> 152; 256 (B8 C2048), T 512 111 -> 121 with four segments: not cut.  bf16 a little more so.
constexpr int V4_MAX_SEG = 64;
struct V4Plan { int nseg, bps; };
static V4Plan v4_plan(int B, int Tlen, int C) {
    const int nblk = (Tlen + CK - 1) / CK, groups = (B * C + 63) / 64, ncu = cu_count();
    const int want = std::min({V4_MAX_SEG, std::max(2 * ncu / groups, std::min(8, 4 * ncu / groups)), nblk / 2});
    if (want < 6 || nblk < 16) return V4Plan{1, nblk};
    const int bps = (nblk + want - 1) / want;
    return V4Plan{(nblk + bps - 1) / bps, bps};
}
size_t v4_checkpoint_bytes(int B, int Tlen, int C) {
    return (size_t)((Tlen + CK - 1) / CK) * 5 * (size_t)B * C * sizeof(float);
}
size_t v4_forward_scratch(int B, int Tlen, int C) {          // the summaries; none where nothing is cut
    const V4Plan pl = v4_plan(B, Tlen, C);
    return pl.nseg > 1 ? (size_t)pl.nseg * 5 * B * C * sizeof(float) : 0;
}
// gw, gu partials of every segment, the summaries, room for checkpoints
size_t v4_backward_workspace(int B, int Tlen, int C) {
    return 2 * (size_t)v4_plan(B, Tlen, C).nseg * B * C * sizeof(float) + v4_forward_scratch(B, Tlen, C) + v4_checkpoint_bytes(B, Tlen, C);
}

// whether the 16-byte fetches apply: a piece of 16 / sizeof(T) chains must not straddle two batch rows, and the
// tensors must be 16-byte aligned
template <class T> static bool v4_wide(int C, std::initializer_list<const void *> tensors) {
    if (C % (16 / (int)sizeof(T)) != 0) return false;
    for (const void *p : tensors)
        if (p && (reinterpret_cast<uintptr_t>(p) & 15u) != 0) return false;
    return true;
}

template <class T> constexpr size_t v4_forward_lds() { return (size_t)V4_GROUPS * 2 * V4_YW * 2 * CK * 64 * sizeof(T); }

template <class T>
static hipError_t fwd(hipStream_t s, int B, int Tlen, int C, const float *td, const float *tf, const void *k,
                      const void *v, const float *s_in, void *y, float *s_out, float *ckpt, float *part) {
    const int BC = B * C;
    if (Tlen == 1 && !ckpt && y) {
        prof_begin(KID_V4_FORWARD, s);
        hipLaunchKernelGGL((v4_decode<T>), dim3((BC + 255) / 256), dim3(256), 0, s, BC, C, td, tf, (const T *)k, (const T *)v, s_in, (T *)y, s_out);
        prof_end(KID_V4_FORWARD, s);
        return hipGetLastError();
    }
    const V4Plan pl = part ? v4_plan(B, Tlen, C) : V4Plan{1, (Tlen + CK - 1) / CK};
    static PerDevice lds_limit;
    const hipError_t lds_ok = lds_limit.once([] {           // (more than the 64 KB a kernel gets by default, for fp32)
        hipError_t e = hipFuncSetAttribute((const void *)v4_forward<T, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)v4_forward_lds<T>());
        if (e == hipSuccess) e = hipFuncSetAttribute((const void *)v4_forward<T, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)v4_forward_lds<T>());
        return e;
    });
    if (lds_ok != hipSuccess) return lds_ok;
    if (pl.nseg > 1)
        hipLaunchKernelGGL((v4_summary_forward<T>), dim3((BC + 63) / 64, (pl.nseg - 1 + SW - 1) / SW), dim3(64 * SW), 0, s, BC, Tlen, C, td,
                           (const T *)k, (const T *)v, part, pl.nseg, pl.bps);
    prof_begin(KID_V4_FORWARD, s);
    const dim3 grid(((BC + 63) / 64 + V4_GROUPS - 1) / V4_GROUPS, pl.nseg), block(64 * (1 + V4_YW) * V4_GROUPS);
    if (v4_wide<T>(C, {k, v, y}))
        hipLaunchKernelGGL((v4_forward<T, true>), grid, block, v4_forward_lds<T>(), s, BC, Tlen, C, td, tf, (const T *)k,
                           (const T *)v, s_in, (T *)y, s_out, ckpt, part, pl.bps);
    else
        hipLaunchKernelGGL((v4_forward<T, false>), grid, block, v4_forward_lds<T>(), s, BC, Tlen, C, td, tf, (const T *)k,
                           (const T *)v, s_in, (T *)y, s_out, ckpt, part, pl.bps);
    prof_end(KID_V4_FORWARD, s);
    return hipGetLastError();
}

template <class T>
static hipError_t bwd(hipStream_t s, int B, int Tlen, int C, const float *td, const float *tf, const void *k,
                      const void *v, const float *s_in, const void *gy, const float *gs_out, float *gtd, float *gtf,
                      void *gk, void *gv, float *gs_in, const float *ckpt, float *ws) {
    const int BC = B * C;
    // (in place, the first segment's workgroups would write the state gradient that the others read)
    const bool cut = !overlap(gs_in, gs_out, (size_t)BC * 3 * sizeof(float));
    const V4Plan pl = cut ? v4_plan(B, Tlen, C) : V4Plan{1, (Tlen + CK - 1) / CK};
    float *gw_part = ws, *gu_part = gw_part + (size_t)pl.nseg * BC, *part = gu_part + (size_t)pl.nseg * BC;
    if (!ckpt) {           // no checkpoints from the forward call: make them now
        float *own = part + (pl.nseg > 1 ? (size_t)pl.nseg * 5 * BC : 0);
        hipError_t e = fwd<T>(s, B, Tlen, C, td, tf, k, v, s_in, nullptr, nullptr, own, pl.nseg > 1 ? part : nullptr);
        if (e != hipSuccess) return e;
        ckpt = own;
    }
    if (pl.nseg > 1)
        hipLaunchKernelGGL((v4_summary_backward<T>), dim3((BC + 63) / 64, (pl.nseg - 1 + SW - 1) / SW), dim3(64 * SW), 0, s, BC, Tlen, C, td, tf,
                           (const T *)k, (const T *)v, (const T *)gy, ckpt, part, pl.nseg, pl.bps);
    prof_begin(KID_V4_BACKWARD, s);
    auto kernel = pl.nseg > 1 || sizeof(T) == 4 ? v4_backward<T, true> : v4_backward<T, sizeof(T) == 4>;
    hipLaunchKernelGGL(kernel, dim3((BC + 63) / 64, pl.nseg), dim3(128), 0, s, BC, Tlen, C, td, tf, (const T *)k, (const T *)v,
                       (const T *)gy, gs_out, ckpt, gw_part, gu_part, (T *)gk, (T *)gv, gs_in, part, pl.bps);
    prof_end(KID_V4_BACKWARD, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(v4_sum, dim3((C + 31) / 32, 2), dim3(256), 0, s, B * pl.nseg, C, gw_part, gu_part, gtd, gtf);
    return hipGetLastError();
}

hipError_t v4_forward_dispatch(hipStream_t s, int dtype, int B, int Tlen, int C, const float *td, const float *tf,
                               const void *k, const void *v, const float *s_in, void *y, float *s_out, float *ckpt, float *part) {
    switch (dtype) {
        case 0: return fwd<float>(s, B, Tlen, C, td, tf, k, v, s_in, y, s_out, ckpt, part);
        case 1: return fwd<bf16>(s, B, Tlen, C, td, tf, k, v, s_in, y, s_out, ckpt, part);
        default: return fwd<f16>(s, B, Tlen, C, td, tf, k, v, s_in, y, s_out, ckpt, part);
    }
}

hipError_t v4_backward_dispatch(hipStream_t s, int dtype, int B, int Tlen, int C, const float *td, const float *tf,
                                const void *k, const void *v, const float *s_in, const void *gy, const float *gs_out,
                                float *gtd, float *gtf, void *gk, void *gv, float *gs_in, const float *ckpt, float *ws) {
    switch (dtype) {
        case 0: return bwd<float>(s, B, Tlen, C, td, tf, k, v, s_in, gy, gs_out, gtd, gtf, gk, gv, gs_in, ckpt, ws);
        case 1: return bwd<bf16>(s, B, Tlen, C, td, tf, k, v, s_in, gy, gs_out, gtd, gtf, gk, gv, gs_in, ckpt, ws);
        default: return bwd<f16>(s, B, Tlen, C, td, tf, k, v, s_in, gy, gs_out, gtd, gtf, gk, gv, gs_in, ckpt, ws);
    }
}

}  // namespace wkv
