// The gated delta rule with a decay per channel: the reference's kda_scan (src/kernels/ops.metal:459-519), the
// recurrence of the linear-attention layers beside attention in Qwen3.5's encoder (src/models/qwen_text.cpp:374-382).
// For each head, with S its 128 x 128 state (stored transposed: state[h][j][i] = S[i][j]) and each token in order:
//   S[i][:] *= exp(g[i]);  delta[j] = (v[j] - sum_i S[i][j] k[i]) * beta
//   S[i][j] += k[i] * delta[j];  o[j] = sum_i S[i][j] q[i] / sqrt(128)
//
// The design is this one's own. Row j of a head's transposed state evolves on its own: it needs the token's shared
// q, k, g and its own v[j]. A row is 16 lanes (one DPP row) of 8 values (lane l: channels 4l .. 4l + 3 and
// 64 + 4l .. 64 + 4l + 3), so the two sums over channels are 8 fused multiply-adds a lane and four v_add_f32_dpp:
// all VALU, no LDS round trip and no barrier inside a token. A workgroup of 4 waves takes 16 rows of one head
// (grid: heads x 8), so 32 heads make 1024 waves, one a SIMD. (The kernel also takes 32-lane rows of 4 values, the
// two DPP rows of a pair added by v_permlane16_swap: twice the waves, a third more instructions a token, slower.)
// Tokens go through LDS in batches of 16, two buffers: the workgroup stages a batch's q, k and exp(g) rows once
// (coalesced 16-byte loads fetched into registers while the previous batch runs; the exponential computed once a
// channel, not once a row), its v and beta; each lane runs the batch's tokens out of LDS (a lane reads its runs of
// a vector as 16-byte reads, a row's lanes reading contiguous 256-byte runs), reading a token's operands one token
// ahead of the state's chain, and the batch's outputs leave as one coalesced store after the next barrier. One
// barrier a batch. The token loop is one basic block: a token's output reduction is issued after the next token's
// state update (it is off the state's chain), the rollback snapshot has a loop of its own for the one batch that
// holds it, and nothing in the loop is conditional.
// Bound: the token recurrence (a dependent chain of decay, dot product, lane reduction and update per token) and
// the VALU (no packed FP32 here): 7 flops a channel a row a token. This is the kernel of short runs, and of calls with no
// workspace; long runs go by chunks of 16 tokens (below).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device.hpp"

namespace mako {
namespace {

constexpr int kD = 128, kBatch = 16;

struct ScanParams {
    const float *q, *k, *v, *g, *beta;
    float* state;
    float* o;
    float* snap_state;
    uint32_t tokens, qkv_stride, inner, heads, snap;
};

// bound_ctrl set: every source lane of these patterns is inside the row, and the compiler then folds the move into
// the add (v_add_f32_dpp).
template <int CTRL>
__device__ __forceinline__ float dpp(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Sum over the LANES lanes of a state row, in every lane: xor 1 and xor 2 within quads, the half-row and row mirrors
// (16 lanes), then, for 32-lane rows, the two 16-lane rows of each pair added by v_permlane16_swap_b32 (with both
// operands x it returns the pair's even row and its odd row in every lane of the pair), a VALU exchange with no
// LDS round trip.
template <int LANES>
__device__ __forceinline__ float row_sum(float x)
{
    x += dpp<0xb1>(x);   // quad_perm [1, 0, 3, 2]
    x += dpp<0x4e>(x);   // quad_perm [2, 3, 0, 1]
    x += dpp<0x141>(x);  // row_half_mirror
    x += dpp<0x140>(x);  // row_mirror
    if (LANES == 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(as_u32(x), as_u32(x), false, false);
        x = __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
    }
    return x;
}

// The LDS of the token-by-token scan: two batch buffers, the next batch's rows are fetched into registers while this
// batch runs out of LDS. (kda_scan_rows has them as arrays of their own: members of one struct cost it 1-2 %.)
using RowsVectors = float[2][kBatch][kD];
template <int LANES>
using RowsValues = float[2][kBatch][256 / LANES];
using RowsBetas = float[2][kBatch];

// LANES lanes a state row, V = 128 / LANES values a lane in G = V / 4 runs of 4 channels: run r of lane l holds
// channels 4 LANES r + 4 l .. + 3, so a run of the lanes of a row is 16 LANES contiguous bytes of a vector. The work of
// threads 0 .. 255 of workgroup (head, rows); the vectors 16-byte aligned.
template <int LANES>
__device__ __forceinline__ void scan_rows(const ScanParams& a, RowsVectors& qs, RowsVectors& ks, RowsVectors& es,
                                          RowsValues<LANES>& vs, RowsBetas& bs, RowsValues<LANES>& os)
{
    constexpr int V = kD / LANES, G = V / 4, ROWS = 256 / LANES;
    const uint32_t tid = threadIdx.x, h = blockIdx.x, j0 = blockIdx.y * ROWS, row = tid / LANES, l = tid % LANES;
    uint32_t ch[G];
    #pragma unroll
    for (int r = 0; r < G; ++r)
        ch[r] = 4 * LANES * r + 4 * l;
    float* mg = a.state + ((size_t)h * kD + j0 + row) * kD;
    float m[V];
    #pragma unroll
    for (int r = 0; r < G; ++r) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(mg + ch[r]);
        for (int n = 0; n < 4; ++n)
            m[4 * r + n] = x[n];
    }
    const float scale = 0.08838834764831845f;  // 1 / sqrt(128)
    const size_t hq = (size_t)h * kD;
    // Staging of a batch: thread tid moves runs tid and tid + 256 (token run / 32, channels 4 (run % 32) ..) of q, k
    // and g, v of (token tid / ROWS, row tid % ROWS) and beta of token tid. Past the last token the loads read the
    // last token again (put skips them): loads issued on every path let the compiler wait for exactly the older
    // memory operations in the token loop, where a load under a branch made it wait for these too.
    struct Stage {
        f32x4 q[2], k[2], g[2];
        float v, b;
    };
    auto fetch = [&](Stage& st, uint32_t t0) __attribute__((always_inline)) {
        const uint32_t last = a.tokens - 1;
        #pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t e = tid + 256 * i, t = min(t0 + (e >> 5), last), c = 4 * (e & 31);
            const size_t qo = (size_t)t * a.qkv_stride + hq + c, go = (size_t)t * a.inner + hq + c;
            st.q[i] = *reinterpret_cast<const f32x4*>(a.q + qo);
            st.k[i] = *reinterpret_cast<const f32x4*>(a.k + qo);
            st.g[i] = *reinterpret_cast<const f32x4*>(a.g + go);
        }
        st.v = a.v[(size_t)min(t0 + tid / ROWS, last) * a.qkv_stride + hq + j0 + tid % ROWS];
        st.b = a.beta[(size_t)min(t0 + tid, last) * a.heads + h];
    };
    auto put = [&](const Stage& st, int b, uint32_t t0) __attribute__((always_inline)) {
        const uint32_t np = min((uint32_t)kBatch, a.tokens - t0);
        #pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t e = tid + 256 * i, tt = e >> 5, c = 4 * (e & 31);
            if (tt < np) {
                *reinterpret_cast<f32x4*>(&qs[b][tt][c]) = st.q[i];
                *reinterpret_cast<f32x4*>(&ks[b][tt][c]) = st.k[i];
                *reinterpret_cast<f32x4*>(&es[b][tt][c]) =
                    f32x4{__expf(st.g[i][0]), __expf(st.g[i][1]), __expf(st.g[i][2]), __expf(st.g[i][3])};
            }
        }
        if (tid < np * ROWS)
            vs[b][tid / ROWS][tid % ROWS] = st.v;
        if (tid < np)
            bs[b][tid] = st.b;
    };
    // One token out of buffer b; the operands of the token are read before the state's chain needs them.
    struct Ops {
        f32x4 e[G], k[G], q[G];
        float v, b;
    };
    auto ops = [&](Ops& x, int b, uint32_t tt) __attribute__((always_inline)) {
        #pragma unroll
        for (int r = 0; r < G; ++r) {
            x.e[r] = *reinterpret_cast<const f32x4*>(&es[b][tt][ch[r]]);
            x.k[r] = *reinterpret_cast<const f32x4*>(&ks[b][tt][ch[r]]);
            x.q[r] = *reinterpret_cast<const f32x4*>(&qs[b][tt][ch[r]]);
        }
        x.v = vs[b][tt][row];
        x.b = bs[b][tt];
    };
    // The state's update by one token; returns this lane's part of the token's output (its channels' terms). SNAP:
    // the batch holds token `snap` - 1, so the state after it is copied out.
    auto state = [&](auto SNAP_, const Ops& x, uint32_t t) __attribute__((always_inline)) {
        constexpr bool SNAP = decltype(SNAP_)::value;
        float ev[V], kv[V], qv[V];
        #pragma unroll
        for (int r = 0; r < G; ++r)
            #pragma unroll
            for (int n = 0; n < 4; ++n) {
                ev[4 * r + n] = x.e[r][n];
                kv[4 * r + n] = x.k[r][n];
                qv[4 * r + n] = x.q[r][n];
            }
        float s0 = 0.0f, s1 = 0.0f;
        #pragma unroll
        for (int n = 0; n < V; n += 2) {
            m[n] *= ev[n];
            m[n + 1] *= ev[n + 1];
            s0 = fmaf(m[n], kv[n], s0);
            s1 = fmaf(m[n + 1], kv[n + 1], s1);
        }
        const float d = (x.v - row_sum<LANES>(s0 + s1)) * x.b;
        float u0 = 0.0f, u1 = 0.0f;
        #pragma unroll
        for (int n = 0; n < V; n += 2) {
            m[n] = fmaf(kv[n], d, m[n]);
            m[n + 1] = fmaf(kv[n + 1], d, m[n + 1]);
            u0 = fmaf(m[n], qv[n], u0);
            u1 = fmaf(m[n + 1], qv[n + 1], u1);
        }
        if (SNAP && t + 1 == a.snap) {  // the state after `snap` tokens (uniform across the workgroup)
            float* sg = a.snap_state + ((size_t)h * kD + j0 + row) * kD;
            #pragma unroll
            for (int r = 0; r < G; ++r)
                *reinterpret_cast<f32x4*>(sg + ch[r]) = f32x4{m[4 * r], m[4 * r + 1], m[4 * r + 2], m[4 * r + 3]};
        }
        return u0 + u1;
    };
    // The token's output: the row's sum of the lanes' parts, into the batch's output buffer.
    auto emit = [&](float u, int b, uint32_t tt) __attribute__((always_inline)) {
        const float out = row_sum<LANES>(u);
        os[b][tt][row] = out * scale;  // every lane of the row holds the same sum
    };
    auto store_out = [&](int b, uint32_t t0) __attribute__((always_inline)) {
        const uint32_t np = min((uint32_t)kBatch, a.tokens - t0);
        if (tid < np * ROWS)
            a.o[(size_t)(t0 + tid / ROWS) * a.inner + hq + j0 + tid % ROWS] = os[b][tid / ROWS][tid % ROWS];
    };
    if (a.tokens > 0) {
        Stage st;
        fetch(st, 0);
        put(st, 0, 0);
        __syncthreads();
        int b = 0;
        for (uint32_t t0 = 0; t0 < a.tokens; t0 += kBatch, b ^= 1) {
            const bool more = t0 + kBatch < a.tokens;
            // The previous batch's outputs (written before the last barrier), stored before the next batch's loads
            // are issued: the token loop reuses the store's registers, and the wait for the store (memory
            // operations complete in order) then leaves the loads in flight.
            if (t0 > 0)
                store_out(b ^ 1, t0 - kBatch);
            if (more)
                fetch(st, t0 + kBatch);  // in flight while this batch runs
            const uint32_t np = min((uint32_t)kBatch, a.tokens - t0);
            auto tokens = [&](auto SNAP) __attribute__((always_inline)) {
                Ops x0, x1;
                ops(x0, b, 0);
                uint32_t tt = 0;
                for (; tt + 1 < np; tt += 2) {  // two tokens a trip: each token's operands read a token ahead
                    ops(x1, b, tt + 1);
                    const float u0 = state(SNAP, x0, t0 + tt);
                    ops(x0, b, min(tt + 2, (uint32_t)kBatch - 1));  // (past the batch: read, not used)
                    const float u1 = state(SNAP, x1, t0 + tt + 1);
                    emit(u0, b, tt);  // off the state's chain: its reduction fills the next token's wait states
                    emit(u1, b, tt + 1);
                }
                if (tt < np)
                    emit(state(SNAP, x0, t0 + tt), b, tt);
            };
            if (a.snap > t0 && a.snap <= t0 + np)
                tokens(std::true_type{});
            else
                tokens(std::false_type{});
            if (more)
                put(st, b ^ 1, t0 + kBatch);  // buffer b ^ 1 was last read before the previous barrier
            __syncthreads();
        }
        store_out(b ^ 1, (a.tokens - 1) / kBatch * kBatch);
    }
    #pragma unroll
    for (int r = 0; r < G; ++r)
        *reinterpret_cast<f32x4*>(mg + ch[r]) = f32x4{m[4 * r], m[4 * r + 1], m[4 * r + 2], m[4 * r + 3]};
}

template <int LANES>
__global__ __launch_bounds__(256) void kda_scan_rows(const ScanParams a)
{
    __shared__ __attribute__((aligned(16))) RowsVectors qs, ks, es;
    __shared__ RowsValues<LANES> vs;
    __shared__ RowsBetas bs;
    __shared__ RowsValues<LANES> os;
    scan_rows<LANES>(a, qs, ks, es, vs, bs, os);
}

constexpr int kScanLanes = 16;  // lanes a state row: 8 values a lane, one wave a SIMD at 32 heads

// ---- long runs: chunks of 16 tokens ------------------------------------------------------------------------------
//
// Token by token the recurrence is a serial chain of ~400 cycles a token on a quarter of the issue slots (4096 tokens of
// 32 heads: 717 us). Over a chunk of 16 tokens with S its first state, E(t, s) the product of the decays of tokens
// s + 1 .. t and Gamma_t that of all up to t (per channel),
//   d = W (v - (Gamma k) S),  o = ((Gamma q) S + B d) / sqrt(128),  S' = Gamma_last S + (E(last, .) k)^T d
//   A[t][s] = k_t . E(t, s) k_s (s < t),  B[t][s] = q_t . E(t, s) k_s (s <= t),  W = (1 + diag(beta) A)^-1 diag(beta)
// (the delta rule's 16 rank-one updates solved at once), which is seven small matrix products. Products of decays are
// formed one factor at a time as the recurrence forms them, never as exponentials of summed logarithms or as ratios:
// no cancellation. Everything is f32, on v_mfma_f32_16x16x4_f32; against 64 bits the outputs are within 1 % of the
// recurrence's error (1.65e-7 against 1.67e-7 over 97 to 3000 tokens), the state closer (1.37e-7 and 1.53e-7: one
// rounding at its size a chunk).
//
// The products take terms the recurrence does not have, times zero: tokens after the output's (W and B above their
// diagonals) and channels whose state is 0. Where all factors are finite that is exact. Where one is not (an input, or a
// product of decays that grow past f32, which may meet a state of 0), the launch's tokens are left to the recurrence:
// kda_chunk marks the chunk, or its d is not finite, and the workgroup, its state not yet stored, takes them by scan_rows.
// A value that is not finite then reaches what it reaches token by token. The output wave looks, off the state's chain
// (on it, a look at d and a way out of the loop took 5 to 9 %).
//
// kda_chunk: a workgroup a (chunk, head) makes everything of a chunk that needs no state, as the LDS image of the next
// kernel's stage (28 KiB in the workspace): Gamma k, Gamma q, E(last, .) k, Gamma_last, W and B.
// kda_scan_chunks: a workgroup a (head, 16 columns of S), the chunks in order. Waves 0 - 3 hold S, 32 channels each, as
// the accumulators of 16 x 16 blocks: register r of lane (g, c) is channel 16 b + 4 g + r of column c, which is also the
// B operand of the products with S when MFMA r takes channels 4 g + r as its k, and likewise d's and v's tokens, so
// nothing moves between lanes. The waves' shares of (Gamma k) S meet in LDS; d is computed by each. Waves 4 and 5 bring
// the images and v in by LDS DMA, three chunks ahead. (A first form made the images in the workgroup, from rows loaded a
// chunk ahead: 2.1 us a chunk, waiting for the loads.)
// A snapshot's token ends a chunk: the chunks of tokens [0, snap) are followed by those of [snap, tokens).
constexpr uint32_t kChunk = 16, kCRow = kD + 4;  // floats a staged row (the pad spreads 16 rows over the banks)

struct ChunkImage {
    float kg[kChunk][kCRow], qg[kChunk][kCRow], ke[kChunk][kCRow];
    float last[kD];
    float w[kChunk][kChunk], b[kChunk][kChunk];
    uint32_t bad;  // something above is not finite
    float pad[191];
};
static_assert(sizeof(ChunkImage) == 28 * 1024, "whole DMA pieces");

struct ChunkParams {
    ScanParams s;
    ChunkImage* image;    // [chunk of the launch][head]
    uint32_t c0, n;       // the launch's chunks, of all
    uint32_t before;      // chunks of [0, snap)
};

// Chunk c's first token and count.
__device__ __forceinline__ void chunk_of(const ChunkParams& a, uint32_t c, uint32_t& t0, uint32_t& np)
{
    t0 = c < a.before ? c * kChunk : a.s.snap + (c - a.before) * kChunk;
    np = min(kChunk, (c < a.before ? a.s.snap : a.s.tokens) - t0);
}

__global__ __launch_bounds__(256) void kda_chunk(const ChunkParams a)
{
    __shared__ __attribute__((aligned(16))) float ks[kChunk][kD], qs[kChunk][kD], es[kChunk][kD];
    __shared__ float as[kChunk][kChunk + 1], bs[kChunk][kChunk + 1], beta[kChunk];
    __shared__ uint32_t bad;
    const uint32_t tid = threadIdx.x, h = blockIdx.x, c = a.c0 + blockIdx.y;
    uint32_t t0, np;
    chunk_of(a, c, t0, np);
    const size_t hq = (size_t)h * kD;
    #pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t e = tid + 256 * i, t = e >> 5, ch = 4 * (e & 31);
        f32x4 k{}, q{}, d{1.0f, 1.0f, 1.0f, 1.0f};
        if (t < np) {
            const size_t qo = (size_t)(t0 + t) * a.s.qkv_stride + hq + ch;
            k = *reinterpret_cast<const f32x4*>(a.s.k + qo);
            q = *reinterpret_cast<const f32x4*>(a.s.q + qo);
            const f32x4 g = *reinterpret_cast<const f32x4*>(a.s.g + (size_t)(t0 + t) * a.s.inner + hq + ch);
            d = f32x4{__expf(g[0]), __expf(g[1]), __expf(g[2]), __expf(g[3])};
        }
        *reinterpret_cast<f32x4*>(&ks[t][ch]) = k;
        *reinterpret_cast<f32x4*>(&qs[t][ch]) = q;
        *reinterpret_cast<f32x4*>(&es[t][ch]) = d;
    }
    if (tid < kChunk)
        beta[tid] = tid < np ? a.s.beta[(size_t)(t0 + tid) * a.s.heads + h] : 0.0f;
    if (tid == 0)
        bad = 0;
    __syncthreads();
    // Row s of 16 lanes, 8 channels a lane: p = E(t, s) k_s, one more factor a step.
    const uint32_t s = tid >> 4, l = tid & 15, first = __builtin_amdgcn_readfirstlane(s);
    const f32x4 one{1.0f, 1.0f, 1.0f, 1.0f};
    f32x4 p0 = *reinterpret_cast<const f32x4*>(&ks[s][4 * l]), p1 = *reinterpret_cast<const f32x4*>(&ks[s][64 + 4 * l]);
    for (uint32_t t = first; t < kChunk; ++t) {
        const f32x4 e0 = *reinterpret_cast<const f32x4*>(&es[t][4 * l]), e1 = *reinterpret_cast<const f32x4*>(&es[t][64 + 4 * l]);
        const f32x4 k0 = *reinterpret_cast<const f32x4*>(&ks[t][4 * l]), k1 = *reinterpret_cast<const f32x4*>(&ks[t][64 + 4 * l]);
        const f32x4 q0 = *reinterpret_cast<const f32x4*>(&qs[t][4 * l]), q1 = *reinterpret_cast<const f32x4*>(&qs[t][64 + 4 * l]);
        p0 *= t > s ? e0 : one;
        p1 *= t > s ? e1 : one;
        float x = 0.0f, y = 0.0f;
        #pragma unroll
        for (int n = 0; n < 4; ++n) {
            x = fmaf(k0[n], p0[n], x);
            y = fmaf(q0[n], p0[n], y);
        }
        #pragma unroll
        for (int n = 0; n < 4; ++n) {
            x = fmaf(k1[n], p1[n], x);
            y = fmaf(q1[n], p1[n], y);
        }
        x = row_sum<16>(x);
        y = row_sum<16>(y);
        as[t][s] = x;             // (used for s < t only)
        bs[t][s] = t >= s ? y : 0.0f;
    }
    for (uint32_t t = 0; t < first; ++t)
        bs[t][s] = 0.0f;
    __syncthreads();
    ChunkImage& out = a.image[(size_t)blockIdx.y * a.s.heads + h];
    float z = 0.0f;  // stays 0 while what is added, times 0, is finite
    {
        // the running products: 128 threads forward, 128 backward, a channel each
        const uint32_t i = tid & 127;
        float p = 1.0f;
        if (tid < 128) {
            #pragma unroll
            for (uint32_t t = 0; t < kChunk; ++t) {
                p *= es[t][i];
                const float kg = p * ks[t][i], qg = p * qs[t][i];
                out.kg[t][i] = kg;
                out.qg[t][i] = qg;
                z = fmaf(kg, 0.0f, fmaf(qg, 0.0f, z));
            }
            out.last[i] = p;
            z = fmaf(p, 0.0f, z);
        } else {
            #pragma unroll
            for (uint32_t n = 0; n < kChunk; ++n) {
                const uint32_t t = kChunk - 1 - n;
                const float ke = p * ks[t][i];
                out.ke[t][i] = ke;
                z = fmaf(ke, 0.0f, z);
                p *= es[t][i];
            }
        }
    }
    if (tid < kChunk) {  // column tid of W by forward substitution
        float w[kChunk];
        #pragma unroll
        for (uint32_t t = 0; t < kChunk; ++t) {
            float x = t == tid ? 1.0f : 0.0f;
            #pragma unroll
            for (uint32_t r = 0; r < t; ++r)
                x = fmaf(-as[t][r], w[r], x);
            w[t] = x * beta[t];
            out.w[t][tid] = w[t];
            z = fmaf(w[t], 0.0f, z);
        }
    }
    const float b = bs[tid >> 4][tid & 15];
    out.b[tid >> 4][tid & 15] = b;
    if (fmaf(b, 0.0f, z) != 0.0f)  // (not a number is not equal to anything)
        bad = 1;
    __syncthreads();
    if (tid == 0)
        out.bad = bad;
}

__device__ __forceinline__ f32x4 mfma4(float x, float y, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }

// 16 bytes a lane from base + off to LDS m0 + 16 lane.
__device__ __forceinline__ void dma16(uint32_t m0, const void* base, uint32_t off)
{
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(m0), "v"(off), "s"(base)
                 : "memory", "m0");
#pragma clang diagnostic pop
}

__global__ __launch_bounds__(448) void kda_scan_chunks(const ChunkParams a)
{
    constexpr uint32_t kSlots = 4, kPieces = sizeof(ChunkImage) / 1024;  // a wave DMAs half the pieces, and v
    struct Stage {
        ChunkImage x;
        float v[kChunk][kChunk];
    };
    __shared__ __attribute__((aligned(1024))) Stage st[kSlots];
    struct RowsLds {
        RowsVectors q, k, e;
        RowsValues<kScanLanes> v, o;
        RowsBetas b;
    };
    static_assert(sizeof(RowsLds) <= sizeof(st) && kD / (256 / kScanLanes) == kD / 16, "scan_rows' LDS and grid");
    __shared__ uint32_t left;                  // the tokens are left to scan_rows
    __shared__ f32x4 pu[4][64], pq[2][4][64];  // the waves' shares of (Gamma k) S and (Gamma q) S
    __shared__ f32x4 pd[2][64];                // d
    const uint32_t tid = threadIdx.x, lane = tid & 63, h = blockIdx.x, j0 = blockIdx.y * 16;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c16 = lane & 15;
    const size_t hq = (size_t)h * kD;
    const float scale = 0.08838834764831845f;  // 1 / sqrt(128)
    if (w == 4 || w == 5) {
        // Chunk n into slot n % kSlots: pieces w - 4, w - 2, .. of the image, and v (both waves, the same bytes: lane 4 t
        // + n takes columns 4 n .. of token t; past a part chunk's end the last token's, whose products are zeros'), so
        // each wave has the same number in flight. Past the last chunk the DMA reads it again (into slots not read).
        const auto issue = [&](uint32_t n) __attribute__((always_inline)) {
            const uint32_t slot = n % kSlots, cc = min(n, a.n - 1);
            uint32_t t0, np;
            chunk_of(a, a.c0 + cc, t0, np);
            const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>(&st[slot]));
            const ChunkImage* im = a.image + ((size_t)cc * a.s.heads + h);
            #pragma unroll
            for (uint32_t i = 0; i < kPieces / 2; ++i) {
                const uint32_t piece = 2 * i + w - 4;
                dma16(__builtin_amdgcn_readfirstlane(lds + 1024 * piece), im, 1024 * piece + 16 * lane);
            }
            const float* v = a.s.v + (size_t)t0 * a.s.qkv_stride + hq + j0;
            dma16(__builtin_amdgcn_readfirstlane(lds + (uint32_t)sizeof(ChunkImage)), v,
                  min(lane >> 2, np - 1) * a.s.qkv_stride * 4 + 16 * (lane & 3));
        };
        for (uint32_t n = 0; n < kSlots - 1; ++n)
            issue(n);
        // the oldest chunk in flight has landed: all but the kSlots - 2 after it
        const auto landed = [] { asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kSlots - 2) * (kPieces / 2 + 1)) : "memory"); };
        landed();
        __syncthreads();
        for (uint32_t c = 0; c < a.n; ++c) {
            issue(c + kSlots - 1);  // (its slot: chunk c - 1's, read last before the barrier that ended it)
            __syncthreads();        // the shares of chunk c
            landed();
            __syncthreads();        // the end of chunk c
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else if (w == 6) {
        // The outputs, a chunk behind the state, so that they are not on its chain (taken by waves 0 - 3 in turn, they
        // were a quarter of a chunk's time).
        __syncthreads();
        float z = 0.0f;  // stays 0 while every d, times 0, is finite
        uint32_t marked = 0;
        for (uint32_t c = 0; c < a.n; ++c) {
            uint32_t t0, np;
            chunk_of(a, a.c0 + c, t0, np);
            const f32x4 br = *reinterpret_cast<const f32x4*>(&st[c % kSlots].x.b[c16][4 * g]);
            marked |= st[c % kSlots].x.bad;
            __syncthreads();
            __syncthreads();  // the end of chunk c (pq and pd are rewritten two chunks on)
            const f32x4 d = pd[c & 1][lane];
            z = fmaf(d[0], 0.0f, fmaf(d[1], 0.0f, fmaf(d[2], 0.0f, fmaf(d[3], 0.0f, z))));
            f32x4 o{};
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                o = mfma4(br[r], d[r], o);
            o += (pq[c & 1][0][lane] + pq[c & 1][1][lane]) + (pq[c & 1][2][lane] + pq[c & 1][3][lane]);
            float* at = a.s.o + (size_t)t0 * a.s.inner + hq + j0 + c16;
            #pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                if (4 * g + r < np)
                    at[(size_t)(4 * g + r) * a.s.inner] = o[r] * scale;
        }
        const bool leave = __ballot(marked || z != 0.0f) != 0;
        left = leave;
        if (leave)  // (scan_rows writes these outputs again)
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        // Channel 32 w + 16 b + 4 g + r of column j0 + c16: state[h][j][i].
        float* mg = a.s.state + ((size_t)h * kD + j0 + c16) * kD + 32 * w + 4 * g;
        f32x4 m[2];
        #pragma unroll
        for (int b = 0; b < 2; ++b)
            m[b] = *reinterpret_cast<const f32x4*>(mg + 16 * b);
        __syncthreads();  // chunk 0 is staged
        for (uint32_t c = 0; c < a.n; ++c) {
            const Stage& s = st[c % kSlots];
            uint32_t t0, np;
            chunk_of(a, a.c0 + c, t0, np);
            // this wave's shares of (Gamma k) S and (Gamma q) S, tokens 4 g + r of column c16: the second while the first
            // goes through LDS
            f32x4 u[2]{}, y[2]{}, kg[2], qg[2], last[2], v;
            float ke[2][4];
            #pragma unroll
            for (int b = 0; b < 2; ++b) {
                kg[b] = *reinterpret_cast<const f32x4*>(&s.x.kg[c16][32 * w + 16 * b + 4 * g]);
                qg[b] = *reinterpret_cast<const f32x4*>(&s.x.qg[c16][32 * w + 16 * b + 4 * g]);
            }
            const f32x4 wr = *reinterpret_cast<const f32x4*>(&s.x.w[c16][4 * g]);
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] = s.v[4 * g + r][c16];
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                #pragma unroll
                for (int b = 0; b < 2; ++b)
                    u[b] = mfma4(kg[b][r], m[b][r], u[b]);
            #pragma unroll
            for (int b = 0; b < 2; ++b) {
                last[b] = *reinterpret_cast<const f32x4*>(&s.x.last[32 * w + 16 * b + 4 * g]);
                #pragma unroll
                for (int r = 0; r < 4; ++r)
                    ke[b][r] = s.x.ke[4 * g + r][32 * w + 16 * b + c16];
            }
            pu[w][lane] = u[0] + u[1];
            __builtin_amdgcn_sched_barrier(0);
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                #pragma unroll
                for (int b = 0; b < 2; ++b)
                    y[b] = mfma4(qg[b][r], m[b][r], y[b]);
            __syncthreads();
            const f32x4 e = v - ((pu[0][lane] + pu[1][lane]) + (pu[2][lane] + pu[3][lane]));
            pq[c & 1][w][lane] = y[0] + y[1];
            f32x4 d{};
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                d = mfma4(wr[r], e[r], d);
            // the update summed by itself: one rounding at the state's size a chunk
            f32x4 n[2]{};
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                #pragma unroll
                for (int b = 0; b < 2; ++b)
                    n[b] = mfma4(ke[b][r], d[r], n[b]);
            if (w == 0)
                pd[c & 1][lane] = d;
            #pragma unroll
            for (int b = 0; b < 2; ++b)
                #pragma unroll
                for (int r = 0; r < 4; ++r)
                    m[b][r] = fmaf(m[b][r], last[b][r], n[b][r]);
            if (a.s.snap && t0 + np == a.s.snap) {
                float* sg = a.s.snap_state + ((size_t)h * kD + j0 + c16) * kD + 32 * w + 4 * g;
                #pragma unroll
                for (int b = 0; b < 2; ++b)
                    *reinterpret_cast<f32x4*>(sg + 16 * b) = m[b];
            }
            __syncthreads();
        }
        __syncthreads();  // wave 6 has seen the last chunk
        if (!__builtin_amdgcn_readfirstlane(left)) {
            #pragma unroll
            for (int b = 0; b < 2; ++b)
                *reinterpret_cast<f32x4*>(mg + 16 * b) = m[b];
            return;
        }
        uint32_t t0, t1, np;
        chunk_of(a, a.c0 + a.n - 1, t1, np);
        t1 += np;
        chunk_of(a, a.c0, t0, np);
        ScanParams r = a.s;
        r.q += (size_t)t0 * r.qkv_stride;
        r.k += (size_t)t0 * r.qkv_stride;
        r.v += (size_t)t0 * r.qkv_stride;
        r.g += (size_t)t0 * r.inner;
        r.o += (size_t)t0 * r.inner;
        r.beta += (size_t)t0 * r.heads;
        r.tokens = t1 - t0;
        r.snap = r.snap > t0 && r.snap <= t1 ? r.snap - t0 : 0;
        RowsLds& lds = *reinterpret_cast<RowsLds*>(&st[0]);
        scan_rows<kScanLanes>(r, lds.q, lds.k, lds.e, lds.v, lds.b, lds.o);
        return;
    }
    __syncthreads();
}

// The workspace a launch's images take at most: longer runs go in several launches, whose images stay in the last-level
// cache (73 chunks of 32 heads: 30 us to make, bound by their traffic, and 81 us to run, 1.1 us a chunk of LDS and barrier
// latencies around 28 MFMAs a wave).
constexpr uint32_t kChunkTokens = 96;
constexpr size_t kChunkBytes = 64u << 20;

uint32_t chunks_of(const mako_scan_args* a)
{
    return (a->snap + kChunk - 1) / kChunk + (a->tokens - a->snap + kChunk - 1) / kChunk;
}

size_t chunk_bytes(const mako_scan_args* a) { return (size_t)a->heads * sizeof(ChunkImage); }

// The chunks of one launch.
uint32_t chunks_a_launch(const mako_scan_args* a)
{
    return (uint32_t)std::min<size_t>({chunks_of(a), std::max<size_t>(1, kChunkBytes / chunk_bytes(a)), 65535});
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace mako

using namespace mako;

namespace {

// Whether the chunks are the faster kernels, by estimates in us of both: an image 0.0124, a chunk 1.1 and a launch 2.3 for
// each round of heads x 8 workgroups over the CUs, against 0.175 a token while those workgroups have a CU each and 0.00375
// a token and head past that (two or three of them share a CU then, and the chunks' one a CU gains less). us, token by
// token / by chunks: 32 heads, 96 tokens 21.2 / 17.1, 200 39 / 26, 1024 182 / 90, 4096 716 / 356; 64 heads, 96 27.1 /
// 26.5, 100 28.1 / 28.9, 1024 245 / 186; 256 heads, 100 98 / 102, 1024 1027 / 918; 512 heads, 200 376 / 452; 1024 heads,
// 100 396 / 632.
bool chunks_take(const mako_scan_args* a)
{
    if (!a->heads || a->tokens < kChunkTokens || a->snap > a->tokens)
        return false;
    const uint32_t cus = device_cus(), n = chunks_of(a), per = chunks_a_launch(a);
    const double groups = 8.0 * a->heads, rounds = std::ceil(groups / (cus ? cus : 256));
    const double chunks = 0.0124 * n * a->heads + rounds * (2.3 * ((n + per - 1) / per) + 1.1 * n);
    return chunks <= a->tokens * std::max(0.175, 0.00375 * a->heads);
}

size_t scan_bytes(const mako_scan_args* a) { return chunks_take(a) ? chunks_a_launch(a) * chunk_bytes(a) : 0; }

int scan_core(const mako_scan_args* a, const float* q, const float* k, const float* v, const float* g,
              const float* beta, float* state, float* o, float* snap_state, const Workspace& work, void* stream)
{
    if (!a || !q || !k || !v || !g || !beta || !state || !o || (a->snap && !snap_state))
        return fail(MAKO_EINVAL, "kda_scan: a null argument");
    if (a->head_dim != kD)
        return fail(MAKO_EUNSUPPORTED, "kda_scan: head_dim %u (must be 128)", a->head_dim);
    if (!a->heads || a->qkv_stride < a->heads * kD || a->inner < a->heads * kD)
        return fail(MAKO_EINVAL, "kda_scan: %u heads of 128 in rows of %u (q, k, v) and %u (g, o)", a->heads,
                    a->qkv_stride, a->inner);
    if (a->qkv_stride % 4 || a->inner % 4 || !al16(q) || !al16(k) || !al16(g) || !al16(state) ||
        (a->snap && !al16(snap_state)))
        return fail(MAKO_EINVAL, "kda_scan: q, k, g and the states must be 16-byte aligned, row strides multiples of 4");
    if (a->snap > a->tokens)
        return fail(MAKO_EINVAL, "kda_scan: a snapshot after %u of %u tokens", a->snap, a->tokens);
    if (a->heads > 65535u)
        return fail(MAKO_EINVAL, "kda_scan: %u heads exceed the grid", a->heads);
    ScanParams p{q, k, v, g, beta, state, o, snap_state, a->tokens, a->qkv_stride, a->inner, a->heads, a->snap};
    const hipStream_t s = static_cast<hipStream_t>(stream);
    // chunks, where there is a workspace to be had (a capture, no memory or a caller's shorter one: token by token), v's
    // rows suit 16-byte DMA from 32-bit offsets, and v and the first state outlast a launch that is left to scan_rows
    const size_t bytes = scan_bytes(a);
    const size_t v_end = (size_t)(a->tokens - 1) * a->qkv_stride + (size_t)a->heads * kD,
                 o_end = (size_t)(a->tokens - 1) * a->inner + (size_t)a->heads * kD;
    if (bytes && al16(v) && a->qkv_stride < (1u << 25) && (o >= v + v_end || v >= o + o_end) &&
        !(a->snap && snap_state == state)) {
        if (ChunkImage* ws = static_cast<ChunkImage*>(work.try_get(kWsScan, bytes, s))) {
            const uint32_t n = chunks_of(a), per = chunks_a_launch(a);
            for (uint32_t c = 0; c < n; c += per) {
                const ChunkParams cp{p, ws, c, std::min(per, n - c), (a->snap + kChunk - 1) / kChunk};
                hipLaunchKernelGGL(kda_chunk, dim3(a->heads, cp.n), dim3(256), 0, s, cp);
                hipLaunchKernelGGL(kda_scan_chunks, dim3(a->heads, kD / 16), dim3(448), 0, s, cp);
            }
            return check_launch("kda_scan");
        }
    }
    hipLaunchKernelGGL(kda_scan_rows<kScanLanes>, dim3(a->heads, kD / (256 / kScanLanes)), dim3(256), 0, s, p);
    return check_launch("kda_scan");
}

}  // namespace

extern "C" size_t mako_kda_scan_workspace(const mako_scan_args* a) { return a ? scan_bytes(a) : 0; }

extern "C" int mako_kda_scan(const mako_scan_args* a, const float* q, const float* k, const float* v, const float* g,
                             const float* beta, float* state, float* o, float* snap_state, void* stream)
{
    return scan_core(a, q, k, v, g, beta, state, o, snap_state, library_workspace(kWsScan, "kda_scan"), stream);
}

extern "C" int mako_kda_scan_ws(const mako_scan_args* a, const float* q, const float* k, const float* v, const float* g,
                                const float* beta, float* state, float* o, float* snap_state, void* workspace,
                                size_t workspace_bytes, void* stream)
{
    return scan_core(a, q, k, v, g, beta, state, o, snap_state,
                     caller_workspace(workspace, workspace_bytes, "kda_scan"), stream);
}
