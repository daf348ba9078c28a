// The output projection after attention: Runtime::proj with BF16 weights (src/gpu/runtime.cpp:164-205), i.e. the
// to_bf16 rounding of the activations (src/kernels/gemm.metal:676-681), the dense BF16 GEMM gemm_dense
// (gemm.metal:251-296) and, with bf16_split_, the remainder's GEMM and add_rows (src/kernels/ops.metal:421-437):
//
//   y[r][c] = sum_j w[c][j] * bf16(x[r][j])  (+ sum_j w[c][j] * bf16(x[r][j] - bf16(x[r][j])) with split)
//
// The design is this one's own. Bound: MFMA (a 4096-token, 4096 x 4096 projection is 137 GFLOP against 67 MB of
// output and 64 MB of operands); the read of w for a few rows. Routes: proj_few (few rows), proj_dma and proj_ring (bf16
// rows, and f32 rows after round_rows), proj_tiles (f32 rows without a workspace to round into). In proj_tiles a workgroup of 4 waves computes a BM x 256 tile of y (BM = 256; 128 with split),
// each wave a (BM / 2) x 128 block as 32 x 32 MFMA blocks (v_mfma_f32_32x32x16_bf16) accumulating in f32.
// 64-wide K chunks of x rows and w rows go through LDS, two buffers with one barrier a chunk; the next chunk waits in
// registers while the current one is multiplied, and is stored, and the one after fetched, behind the first MFMAs. Both operands are K-contiguous rows, so every 16-byte run of a row
// is one MFMA operand (8 consecutive k). LDS rows are 128 bytes; the 16-byte run c of row r sits at position
// c ^ ((r / 2) % 8), so the 16 lanes of a ds_read_b128 (16 consecutive rows, one run) and of a ds_write_b128 (two
// rows, eight runs) hit 64 distinct banks. f32 activations are rounded to bf16 (to nearest even) as they are
// staged: the reference's separate to_bf16 pass (and its bf16 copy of x in HBM) is gone.
#include <algorithm>
#include <type_traits>

#include "device.hpp"

namespace mako {
namespace {

constexpr int kBN = 256, kBK = 64;

struct ProjParams {
    const __bf16* w;  // [n][k]
    const void* x;    // [t][ldx], bf16 or f32
    float* y;         // [t][ldy]
    uint32_t t, k, n, ldy, ldx;
    uint32_t tiles_m, tiles_n, tiles, per_xcd;
    uint32_t planes;  // bf16 x of the DMA kernels: 2 when a row's k values come after its k remainders (ldx covers both)
};

// Tile q of the output walks bands of 4 tile rows column by column, and XCD x takes tiles x * per_xcd .. (workgroup
// L runs on XCD L % 8): with 16 x 16 tiles each XCD holds a 4 x 8 block, sharing 4 row panels of x and 8 of w in
// its L2.
__device__ __forceinline__ bool tile_of(const ProjParams& a, uint32_t& tm, uint32_t& tn)
{
    const uint32_t L = blockIdx.x, slot = L >> 3;
    const uint32_t q = (L & 7u) * a.per_xcd + slot;
    if (slot >= a.per_xcd || q >= a.tiles)
        return false;
    const uint32_t band = q / (4u * a.tiles_n), h = min(4u, a.tiles_m - 4u * band), in = q - band * 4u * a.tiles_n;
    tn = in / h;
    tm = 4u * band + in % h;
    return true;
}

__device__ __forceinline__ uint32_t lds_pos(uint32_t row, uint32_t run) { return row * kBK + ((run ^ ((row >> 1) & 7u)) << 3); }

template <int BM, bool XF32, bool SPLIT>
__global__ __launch_bounds__(256, 1) void proj_tiles(const ProjParams a)
{
    constexpr int MB = BM / 64;     // 32-row blocks of x a wave
    constexpr int RA = BM / 32;     // staging rounds of x rows (32 rows a round)
    constexpr int RB = kBN / 32;    // staging rounds of w rows
    __shared__ __attribute__((aligned(16))) __bf16 as[2][BM * kBK];
    __shared__ __attribute__((aligned(16))) __bf16 al[SPLIT ? 2 : 1][SPLIT ? BM * kBK : 8];
    __shared__ __attribute__((aligned(16))) __bf16 bs[2][kBN * kBK];
    uint32_t tm, tn;
    if (!tile_of(a, tm, tn))
        return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 5, c32 = lane & 31;
    const uint32_t t0 = tm * BM, n0 = tn * kBN;
    // staging: thread tid moves run tid % 8 (8 values of k) of rows tid / 8 + 32 i; rows past t / n read the last
    // row (their results are not stored)
    const uint32_t sr = tid >> 3, run = tid & 7;
    uint32_t xo[RA], wo[RB];
    #pragma unroll
    for (int i = 0; i < RA; ++i)
        xo[i] = min(t0 + sr + 32u * i, a.t - 1) * a.ldx + 8 * run;
    #pragma unroll
    for (int i = 0; i < RB; ++i)
        wo[i] = min(n0 + sr + 32u * i, a.n - 1) * a.k + 8 * run;
    struct Stage {
        f32x4 xf[XF32 ? 2 * RA : 1];  // f32 activations, loaded as float vectors (see put)
        u32x4 x[XF32 ? 1 : RA];
        u32x4 w[RB];
    };
    auto fetch = [&](Stage& st, uint32_t k0) __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < RA; ++i) {
            if (XF32) {
                const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.x) + (size_t)xo[i] + k0);
                st.xf[2 * i] = p[0];
                st.xf[2 * i + 1] = p[1];
            } else {
                st.x[i] = *reinterpret_cast<const u32x4*>(static_cast<const __bf16*>(a.x) + (size_t)xo[i] + k0);
            }
        }
        #pragma unroll
        for (int i = 0; i < RB; ++i)
            st.w[i] = *reinterpret_cast<const u32x4*>(a.w + (size_t)wo[i] + k0);
    };
    auto put = [&](const Stage& st, int b) __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < RA; ++i) {
            const uint32_t p = lds_pos(sr + 32u * i, run);
            if (XF32) {
                // Floats come straight from float vectors: hipcc (ROCm 7.2) miscompiles the bf16 packing of
                // floats bit-cast one by one out of a u32x4 (one source converted twice, the loads overlapped).
                const f32x4 v0 = st.xf[2 * i], v1 = st.xf[2 * i + 1];
                const float f[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                u32x4 hi, lo;
                #pragma unroll
                for (int e = 0; e < 4; ++e) {
                    hi[e] = Elem<__bf16>::pack2(f[2 * e], f[2 * e + 1]);
                    if (SPLIT)  // bf16(x - float(bf16(x))), the remainder the reference's bf16_lo keeps
                        lo[e] = Elem<__bf16>::pack2(f[2 * e] - (float)(__bf16)f[2 * e],
                                                    f[2 * e + 1] - (float)(__bf16)f[2 * e + 1]);
                }
                *reinterpret_cast<u32x4*>(as[b] + p) = hi;
                if (SPLIT)
                    *reinterpret_cast<u32x4*>(al[b] + p) = lo;
            } else {
                *reinterpret_cast<u32x4*>(as[b] + p) = st.x[i];
            }
        }
        #pragma unroll
        for (int i = 0; i < RB; ++i)
            *reinterpret_cast<u32x4*>(bs[b] + lds_pos(sr + 32u * i, run)) = st.w[i];
    };
    f32x16 acc[MB][4];
    #pragma unroll
    for (int bi = 0; bi < MB; ++bi)
        #pragma unroll
        for (int bj = 0; bj < 4; ++bj)
            acc[bi][bj] = f32x16{};
    const uint32_t ra = (w >> 1) * (BM / 2), rb = (w & 1) * 128;  // this wave's first x row and w row in the tile
    struct Frag {
        bf16x8 x[MB], xl[SPLIT ? MB : 1], w[4];
    };
    auto read = [&](Frag& f, int b, int kk) __attribute__((always_inline)) {
        const uint32_t rn = 2 * kk + g;
        #pragma unroll
        for (int bi = 0; bi < MB; ++bi) {
            const uint32_t p = lds_pos(ra + 32 * bi + c32, rn);
            f.x[bi] = *reinterpret_cast<const bf16x8*>(as[b] + p);
            if (SPLIT)
                f.xl[bi] = *reinterpret_cast<const bf16x8*>(al[b] + p);
        }
        #pragma unroll
        for (int bj = 0; bj < 4; ++bj)
            f.w[bj] = *reinterpret_cast<const bf16x8*>(bs[b] + lds_pos(rb + 32 * bj + c32, rn));
    };
    auto mfmas = [&](const Frag& f) __attribute__((always_inline)) {
        #pragma unroll
        for (int bi = 0; bi < MB; ++bi)
            #pragma unroll
            for (int bj = 0; bj < 4; ++bj) {
                acc[bi][bj] = Elem<__bf16>::mfma32(f.x[bi], f.w[bj], acc[bi][bj]);
                if (SPLIT)
                    acc[bi][bj] = Elem<__bf16>::mfma32(f.xl[bi], f.w[bj], acc[bi][bj]);
            }
    };
    // One K chunk out of buffer b: the operands of step kk + 1 are read while step kk's MFMAs run, and between(kk)
    // (the staging of a later chunk) is issued behind step kk's MFMAs.
    // sched_barrier keeps each read group ahead of the MFMAs it overlaps (the scheduler otherwise sinks the reads to
    // their first use and the MFMAs wait for LDS).
    auto chunk = [&](int b, auto between) __attribute__((always_inline)) {
        Frag f0, f1;
        read(f0, b, 0);
        read(f1, b, 1);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(f0);
        between(0);
        __builtin_amdgcn_sched_barrier(0);
        read(f0, b, 2);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(f1);
        between(1);
        __builtin_amdgcn_sched_barrier(0);
        read(f1, b, 3);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(f0);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(f1);
    };
    const uint32_t nk = a.k / kBK;
    Stage st;
    fetch(st, 0);
    put(st, 0);
    if (nk > 1)
        fetch(st, kBK);
    __syncthreads();
    uint32_t j = 0;
    for (; j + 2 < nk; ++j) {  // chunk j + 1 goes to the other buffer (last read before the previous barrier)
        const int b = j & 1;
        chunk(b, [&](int kk) __attribute__((always_inline)) {
            if (kk == 0)
                put(st, b ^ 1);
            else
                fetch(st, (j + 2) * kBK);
        });
        __syncthreads();
    }
    if (j + 1 < nk) {
        const int b = j & 1;
        chunk(b, [&](int kk) __attribute__((always_inline)) {
            if (kk == 0)
                put(st, b ^ 1);
        });
        __syncthreads();
        ++j;
    }
    chunk(j & 1, [](int) {});
    // acc[bi][bj] register r of lane (c32, g): row t0 + ra + 32 bi + 8 (r / 4) + 4 g + r % 4, column n0 + rb + 32 bj + c32
    #pragma unroll
    for (int bj = 0; bj < 4; ++bj) {
        const uint32_t c = n0 + rb + 32 * bj + c32;
        if (c >= a.n)
            continue;
        #pragma unroll
        for (int bi = 0; bi < MB; ++bi)
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = t0 + ra + 32 * bi + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row < a.t)
                    a.y[(size_t)row * a.ldy + c] = acc[bi][bj][r];
            }
    }
}

// A raw buffer descriptor over the rows of a tile's panel from `base` (rows of ld values, `rows` of them left in the
// operand): reads at or past the end return zeros.
__device__ __forceinline__ u32x4 panel_rsrc(const __bf16* base, uint32_t rows, uint32_t ld)
{
    const uint64_t a = reinterpret_cast<uint64_t>(base), bytes = (uint64_t)rows * ld * 2;
    return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, (uint32_t)min(bytes, (uint64_t)0xffffffffu), 0x00020000u};
}

// bf16 activations: both operands go global -> LDS by the LDS DMA (buffer_load_dwordx4 ... lds: lane l of a wave
// writes 16 bytes at the wave's LDS base + 16 l, from any offset of its choosing in the tile's panel), with no
// register staging. A stage holds 64 K values of the tile's 256 x rows and 256 w rows (128 bytes a row, so the DMA of
// a row reads whole 128-byte lines; 32-wide stages, which read half lines, ran 3 % slower), two stages (128 KB), one
// barrier a stage: the DMA of stage q + 1 goes out in the first 16 MFMA slots after barrier q, the fragment reads one
// every other slot, a K step ahead of their MFMAs. LDS rows are 128 bytes; the 16-byte run c of row r sits at
// position c ^ ((r / 2) % 8), so the 16 lanes of a ds_read_b128 (16 consecutive rows, one run) hit 64 distinct banks.
// A DMA instruction writes 8 rows (1 KB), lane l taking row l / 8 at position l % 8.
constexpr int kEK = 64;

__device__ __forceinline__ uint32_t epos(uint32_t row, uint32_t run) { return row * kEK + ((run ^ ((row >> 1) & 7u)) << 3); }

// The DMA is issued as inline asm: the compiler, seeing the builtin, waits for every DMA in flight before any LDS read
// (it cannot tell the stages apart). Here the only waits are the stage barriers'. M0 (the DMA's LDS base) is listed as
// clobbered; nothing else in these kernels uses it.
__device__ __forceinline__ void dma_lds(uint32_t voff, uint32_t soff, u32x4 rs, uint32_t lds)
{
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(rs),
                 "s"(__builtin_amdgcn_readfirstlane(soff))
                 : "memory", "m0");
#pragma clang diagnostic pop
}

__global__ __launch_bounds__(256, 1) void proj_dma(const ProjParams a)
{
    __shared__ __attribute__((aligned(16))) __bf16 as[2][kBN * kEK];
    __shared__ __attribute__((aligned(16))) __bf16 bs[2][kBN * kEK];
    uint32_t tm, tn;
    if (!tile_of(a, tm, tn))
        return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 5, c32 = lane & 31;
    const uint32_t t0 = tm * kBN, n0 = tn * kBN;
    const __bf16* x = static_cast<const __bf16*>(a.x);
    uint32_t xo[8], wo[8];
    #pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t row = 64 * w + 8 * i + (lane >> 3), run = (lane & 7) ^ ((row >> 1) & 7);
        xo[i] = (min(t0 + row, a.t - 1) - t0) * a.ldx * 2 + 16 * run;
        wo[i] = (min(n0 + row, a.n - 1) - n0) * a.k * 2 + 16 * run;
    }
    const u32x4 xrs = panel_rsrc(x + (size_t)t0 * a.ldx, a.t - t0, a.ldx);
    const u32x4 wrs = panel_rsrc(a.w + (size_t)n0 * a.k, a.n - n0, a.k);
    const uint32_t wl = __builtin_amdgcn_readfirstlane(64 * w * kEK * 2);  // this wave's first row, LDS bytes
    const uint32_t nk = a.k / kEK, nq = nk * a.planes;  // K stages of w (>= 1), and of x's planes
    const uint32_t abase = (uint32_t)(uintptr_t)&as[0][0] + wl, bbase = (uint32_t)(uintptr_t)&bs[0][0] + wl;
    // DMA instruction i (0 .. 15) of K stage q (values 64 q .. 64 q + 63) into LDS stage q % 2: x piece i / 2 (8 rows)
    // for even i, w piece i / 2 for odd
    auto dma1 = [&](uint32_t q, int i) __attribute__((always_inline)) {
        const uint32_t so = 2 * kEK * q, st = (q & 1) * (kBN * kEK * 2) + 1024 * (i / 2);
        if (i % 2 == 0)
            dma_lds(xo[i / 2], so, xrs, abase + st);
        else
            dma_lds(wo[i / 2], q < nk ? so : so - 2 * a.k, wrs, bbase + st);
    };
    f32x16 acc[4][4];
    #pragma unroll
    for (int bi = 0; bi < 4; ++bi)
        #pragma unroll
        for (int bj = 0; bj < 4; ++bj)
            acc[bi][bj] = f32x16{};
    const uint32_t ra = (w >> 1) * 128, rb = (w & 1) * 128;
    struct Frag {
        bf16x8 x[4], w[4];
    };
    // pieces 0 .. 7 of a fragment: x0, w0, w1, w2, w3, x1, x2, x3, the order the MFMAs (bi outer, bj inner) use them
    auto read1 = [&](Frag& f, uint32_t st, int kk, int piece) __attribute__((always_inline)) {
        const uint32_t rn = 2 * kk + g;
        if (piece == 0 || piece >= 5) {
            const int bi = piece == 0 ? 0 : piece - 4;
            f.x[bi] = *reinterpret_cast<const bf16x8*>(as[st] + epos(ra + 32 * bi + c32, rn));
        } else {
            const int bj = piece - 1;
            f.w[bj] = *reinterpret_cast<const bf16x8*>(bs[st] + epos(rb + 32 * bj + c32, rn));
        }
    };
    // 16 MFMAs on `use`; the reads of `next` (LDS stage st, K step kk of its four) on the even slots; with DMA, the 16
    // instructions of K stage q, one a slot
    auto half = [&](const Frag& use, Frag& next, uint32_t st, int kk, auto DMA, uint32_t q) __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < 16; ++i) {
            acc[i / 4][i % 4] = Elem<__bf16>::mfma32(use.x[i / 4], use.w[i % 4], acc[i / 4][i % 4]);
            __builtin_amdgcn_sched_barrier(0);
            if (i % 2 == 0 && kk >= 0)
                read1(next, st, kk, i / 2);
            if constexpr (decltype(DMA)::value)
                dma1(q, i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using Y = std::true_type;
    using N = std::false_type;
    Frag fa, fb;
    #pragma unroll
    for (int i = 0; i < 16; ++i)
        dma1(0, i);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    #pragma unroll
    for (int i = 0; i < 8; ++i)
        read1(fa, 0, 0, i);
    if (nq > 1) {
        #pragma unroll
        for (int i = 0; i < 16; ++i)
            dma1(1, i);
    }
    __builtin_amdgcn_sched_barrier(0);
    half(fa, fb, 0, 1, N{}, 0);
    half(fb, fa, 0, 2, N{}, 0);
    half(fa, fb, 0, 3, N{}, 0);
    // K stage q: its LDS stage has landed (this wave's DMA by the wait, every wave's by the barrier) and the reads of
    // stage q - 1 are done, so stage q + 1 goes to the other LDS stage while the last K step of q - 1 and the first
    // three of q run. The last K stage has nothing to fetch.
    uint32_t q = 1;
    for (; q + 1 < nq; ++q) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t st = q & 1;
        half(fb, fa, st, 0, Y{}, q + 1);
        half(fa, fb, st, 1, N{}, 0);
        half(fb, fa, st, 2, N{}, 0);
        half(fa, fb, st, 3, N{}, 0);
    }
    if (q < nq) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t st = q & 1;
        half(fb, fa, st, 0, N{}, 0);
        half(fa, fb, st, 1, N{}, 0);
        half(fb, fa, st, 2, N{}, 0);
        half(fa, fb, st, 3, N{}, 0);
    }
    half(fb, fa, 0, -1, N{}, 0);
    #pragma unroll
    for (int bj = 0; bj < 4; ++bj) {
        const uint32_t c = n0 + rb + 32 * bj + c32;
        if (c >= a.n)
            continue;
        #pragma unroll
        for (int bi = 0; bi < 4; ++bi)
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = t0 + ra + 32 * bi + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row < a.t)
                    a.y[(size_t)row * a.ldy + c] = acc[bi][bj][r];
            }
    }
}

// The same in smaller tiles, for calls that make too few 256 x 256 ones for the chip: BM x BN a workgroup, 2 x 2 waves
// of BM / 2 x BN / 2, and a ring of NST K stages, since a small tile multiplies a stage in less time than its DMA takes
// to land: after barrier q, stage q + NST - 1 goes out into the slot stage q - 1 left, and the wait before the barrier
// leaves the NST - 2 stages after q in flight. Past the last stage the DMA reads it again (into slots nothing reads any
// more), so the waits' counts hold to the end; the last ones land before the wave ends.
template <int BM, int BN, int NST>
__global__ __launch_bounds__(256, 1) void proj_ring(const ProjParams a)
{
    constexpr int MB = BM / 64, NB = BN / 64, NM = MB * NB, NR = MB + NB, XD = BM / 32, ND = XD + BN / 32;
    constexpr uint32_t kStage = (BM + BN) * kEK;  // values a stage: BM x rows, then BN w rows
    __shared__ __attribute__((aligned(16))) __bf16 lds[NST * kStage];
    uint32_t tm, tn;
    if (!tile_of(a, tm, tn))
        return;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 5, c32 = lane & 31;
    const uint32_t t0 = tm * BM, n0 = tn * BN;
    // this wave's DMA instructions of a stage: 8 rows each, x's then w's
    uint32_t off[ND];
    #pragma unroll
    for (int i = 0; i < ND; ++i) {
        const bool x = i < XD;
        const uint32_t row = 8 * (x ? XD * w + i : (ND - XD) * w + i - XD) + (lane >> 3), run = (lane & 7) ^ ((row >> 1) & 7);
        off[i] = (x ? (min(t0 + row, a.t - 1) - t0) * a.ldx : (min(n0 + row, a.n - 1) - n0) * a.k) * 2 + 16 * run;
    }
    const u32x4 xrs = panel_rsrc(static_cast<const __bf16*>(a.x) + (size_t)t0 * a.ldx, a.t - t0, a.ldx);
    const u32x4 wrs = panel_rsrc(a.w + (size_t)n0 * a.k, a.n - n0, a.k);
    const uint32_t base = (uint32_t)(uintptr_t)lds;
    const uint32_t xl = __builtin_amdgcn_readfirstlane(base + 1024 * XD * w);
    const uint32_t wl = __builtin_amdgcn_readfirstlane(base + 1024 * (BM / 8 + (ND - XD) * w));
    const uint32_t nk = a.k / kEK, nq = nk * a.planes;
    auto dma1 = [&](uint32_t q, uint32_t slot, int i) __attribute__((always_inline)) {
        const uint32_t st = 2 * kStage * slot;
        if (i < XD)
            dma_lds(off[i], 2 * kEK * q, xrs, xl + st + 1024 * i);
        else
            dma_lds(off[i], 2 * kEK * (q < nk ? q : q - nk), wrs, wl + st + 1024 * (i - XD));
    };
    f32x16 acc[NM];
    #pragma unroll
    for (int i = 0; i < NM; ++i)
        acc[i] = f32x16{};
    const uint32_t ra = (w >> 1) * (BM / 2), rb = BM + (w & 1) * (BN / 2);
    struct Frag {
        bf16x8 f[NR];  // x's MB blocks, then w's NB
    };
    auto read1 = [&](Frag& f, uint32_t slot, int kk, int i) __attribute__((always_inline)) {
        const uint32_t row = (i < MB ? ra + 32 * i : rb + 32 * (i - MB)) + c32;
        f.f[i] = *reinterpret_cast<const bf16x8*>(lds + slot * kStage + epos(row, 2 * kk + g));
    };
    // one K step's MFMAs on `use`, with the reads of `next` (slot, K step kk; kk < 0: none) and, with DMA, stage q's
    // instructions spread between them
    auto step = [&](const Frag& use, Frag& next, uint32_t slot, int kk, auto DMA, uint32_t q, uint32_t to)
        __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < NM; ++i) {
            acc[i] = Elem<__bf16>::mfma32(use.f[i / NB], use.f[MB + i % NB], acc[i]);
            __builtin_amdgcn_sched_barrier(0);
            if (kk >= 0)
                #pragma unroll
                for (int r = i * NR / NM; r < (i + 1) * NR / NM; ++r)
                    read1(next, slot, kk, r);
            if constexpr (decltype(DMA)::value)
                #pragma unroll
                for (int d = i * ND / NM; d < (i + 1) * ND / NM; ++d)
                    dma1(q, to, d);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using Y = std::true_type;
    using N = std::false_type;
    #pragma unroll
    for (int q = 0; q < NST - 1; ++q)
        #pragma unroll
        for (int i = 0; i < ND; ++i)
            dma1(min((uint32_t)q, nq - 1), q, i);
    Frag fa, fb;
    #pragma unroll
    for (int i = 0; i < NR; ++i)
        fb.f[i] = bf16x8{};  // (the first "last K step of the stage before": zeros)
    uint32_t slot = 0, prev = NST - 1;
    for (uint32_t q = 0; q < nq; ++q) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NST - 2) * ND) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        step(fb, fa, slot, 0, Y{}, min(q + NST - 1, nq - 1), prev);
        step(fa, fb, slot, 1, N{}, 0, 0);
        step(fb, fa, slot, 2, N{}, 0, 0);
        step(fa, fb, slot, 3, N{}, 0, 0);
        prev = slot;
        slot = slot + 1 == NST ? 0 : slot + 1;
    }
    step(fb, fa, 0, -1, N{}, 0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    #pragma unroll
    for (int bj = 0; bj < NB; ++bj) {
        const uint32_t c = n0 + (w & 1) * (BN / 2) + 32 * bj + c32;
        if (c >= a.n)
            continue;
        #pragma unroll
        for (int bi = 0; bi < MB; ++bi)
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t row = t0 + ra + 32 * bi + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row < a.t)
                    a.y[(size_t)row * a.ldy + c] = acc[bi * NB + bj][r];
            }
    }
}

// f32 rows rounded to bf16 once, for the DMA kernels (with SPLIT a row's remainders precede its k values: added
// first, they meet small sums; after them, the error against 64 bits was 7.0e-7 at k = 4096 where the two products
// interleaved gave 5.7e-7). Eight values a thread, streamed; bound by HBM (100 MB in 17.6 us at 4096 x 4096, 5.7 TB/s). Rounding in the tiles' staging repeats
// the work and the 32-bit reads in every column of tiles and goes through registers: 167 us at 4096 x 4096, against 129
// for this pass and the DMA kernel (with the split 269 and 233; t = 300: 133 and 28).
template <bool SPLIT>
__global__ __launch_bounds__(256) void round_rows(const float* __restrict__ x, __bf16* __restrict__ out, uint32_t t,
                                                  uint32_t k, uint32_t ldx)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint32_t row = (uint32_t)(i / (k / 8)), c = 8 * (uint32_t)(i % (k / 8));
    if (row >= t)
        return;
    const f32x4* p = reinterpret_cast<const f32x4*>(x + (size_t)row * ldx + c);
    const f32x4 v0 = __builtin_nontemporal_load(p), v1 = __builtin_nontemporal_load(p + 1);
    const float f[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
    u32x4 hi, lo;
    #pragma unroll
    for (int e = 0; e < 4; ++e) {
        hi[e] = Elem<__bf16>::pack2(f[2 * e], f[2 * e + 1]);
        if (SPLIT)
            lo[e] = Elem<__bf16>::pack2(f[2 * e] - (float)(__bf16)f[2 * e], f[2 * e + 1] - (float)(__bf16)f[2 * e + 1]);
    }
    __bf16* o = out + (size_t)row * k * (SPLIT ? 2 : 1) + c;
    *reinterpret_cast<u32x4*>(o + (SPLIT ? k : 0)) = hi;
    if (SPLIT)
        *reinterpret_cast<u32x4*>(o) = lo;
}

// A few rows of x (decode, short verification steps): t <= 16 TB. Bound: the read of w (33.6 MB at 4096 x 4096). A
// 256 x 256 tile a workgroup leaves n / 256 workgroups for the whole chip (16 at n = 4096), so here a workgroup of 8
// waves takes 16 rows of w and all of x, and the waves take every eighth 64-wide K chunk: together they read 1 KiB runs
// of each row, and one round trip covers most of a wave's share. w and x go from memory into the operands of
// v_mfma_f32_16x16x32_bf16 with no LDS: lane (r, g) holds k values 16 g .. 16 g + 15 of a chunk's row r, as two 16-byte
// runs (both operands permute k alike, so a row's 128-byte line is read whole). The waves' partial tiles meet in LDS.
// The next U chunks are loaded while the current U are multiplied. w is read once and streams past the caches; x
// stays in L2 for all workgroups. 4096 x 4096, bf16 x: 77 -> 10.0 us at t = 1 (3.4 TB/s, launch included), 78 -> 15.6
// at t = 32; f32 x 121 -> 10.7 and 24; 2048 x 1024 at t = 1 43 -> 7.2. With more rows every workgroup's own read of x
// from L2 outweighs w's.
constexpr int kFewWaves = 8;
constexpr uint32_t kFewRows = 64;  // at most
constexpr uint32_t kFewBf16 = 32, kFewF32 = 24, kFewSplit = 48;  // where the tiles' kernels can take the rows too (few_takes)

typedef __attribute__((address_space(1))) const u32x4 global_u32x4;

template <int TB, bool XF32, bool SPLIT>
__global__ __launch_bounds__(64 * kFewWaves) void proj_few(const ProjParams a)
{
    constexpr int U = TB == 1 ? 4 : TB == 2 ? 2 : 1;
    __shared__ float part[kFewWaves][TB][16][17];  // [wave][block][row of x][column], padded
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, r = lane & 15;
    const uint32_t n0 = blockIdx.x * 16;
    const __bf16* wp = a.w + (size_t)min(n0 + r, a.n - 1) * a.k + 16 * g;
    size_t xo[TB];
    #pragma unroll
    for (int b = 0; b < TB; ++b)  // rows past t repeat the last one; their results are not stored
        xo[b] = (size_t)min(16u * b + r, a.t - 1) * a.ldx + 16 * g;
    struct Chunk {
        u32x4 w[U][2];
        u32x4 x[U][TB][XF32 ? 1 : 2];
        f32x4 xf[U][TB][XF32 ? 4 : 1];
    };
    const uint32_t nk = a.k / 64;
    // chunks past the end re-read the last one (multiplied only where they exist)
    auto load = [&](Chunk& c, uint32_t q) __attribute__((always_inline)) {
        #pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t k0 = 64 * (size_t)min(q + kFewWaves * u, nk - 1);
            c.w[u][0] = __builtin_nontemporal_load(reinterpret_cast<global_u32x4*>((uintptr_t)(wp + k0)));
            c.w[u][1] = __builtin_nontemporal_load(reinterpret_cast<global_u32x4*>((uintptr_t)(wp + k0 + 8)));
            #pragma unroll
            for (int b = 0; b < TB; ++b) {
                if (XF32) {
                    const f32x4* p = reinterpret_cast<const f32x4*>(static_cast<const float*>(a.x) + xo[b] + k0);
                    #pragma unroll
                    for (int i = 0; i < 4; ++i)
                        c.xf[u][b][i] = p[i];
                } else {
                    const u32x4* p = reinterpret_cast<const u32x4*>(static_cast<const __bf16*>(a.x) + xo[b] + k0);
                    c.x[u][b][0] = p[0];
                    c.x[u][b][1] = p[1];
                }
            }
        }
    };
    f32x4 acc[TB];
    #pragma unroll
    for (int b = 0; b < TB; ++b)
        acc[b] = f32x4{};
    auto mul = [&](const Chunk& c, uint32_t q) __attribute__((always_inline)) {
        #pragma unroll
        for (int u = 0; u < U; ++u) {
            if (q + kFewWaves * u >= nk)
                break;
            #pragma unroll
            for (int b = 0; b < TB; ++b)
                #pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bf16x8 wv = __builtin_bit_cast(bf16x8, c.w[u][h]);
                    u32x4 hi, lo;
                    if (XF32) {
                        const f32x4 v0 = c.xf[u][b][2 * h], v1 = c.xf[u][b][2 * h + 1];
                        const float f[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                        #pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            hi[e] = Elem<__bf16>::pack2(f[2 * e], f[2 * e + 1]);
                            if (SPLIT)
                                lo[e] = Elem<__bf16>::pack2(f[2 * e] - (float)(__bf16)f[2 * e],
                                                            f[2 * e + 1] - (float)(__bf16)f[2 * e + 1]);
                        }
                    } else {
                        hi = c.x[u][b][h];
                    }
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, __builtin_bit_cast(bf16x8, hi), acc[b], 0, 0, 0);
                    if (SPLIT)
                        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, __builtin_bit_cast(bf16x8, lo), acc[b], 0, 0, 0);
                }
        }
    };
    Chunk c0, c1;
    uint32_t q = w;
    if (q < nk) {
        load(c0, q);
        while (true) {
            load(c1, q + kFewWaves * U);
            __builtin_amdgcn_sched_barrier(0);
            mul(c0, q);
            q += kFewWaves * U;
            if (q >= nk)
                break;
            load(c0, q + kFewWaves * U);
            __builtin_amdgcn_sched_barrier(0);
            mul(c1, q);
            q += kFewWaves * U;
            if (q >= nk)
                break;
        }
    }
    // acc[b] register e of lane (r, g): row 16 b + r of x, column n0 + 4 g + e
    #pragma unroll
    for (int b = 0; b < TB; ++b)
        #pragma unroll
        for (int e = 0; e < 4; ++e)
            part[w][b][r][4 * g + e] = acc[b][e];
    __syncthreads();
    for (uint32_t i = tid; i < TB * 256; i += 64 * kFewWaves) {
        const uint32_t row = i >> 4, c = i & 15;
        float s = 0;
        #pragma unroll
        for (int v = 0; v < kFewWaves; ++v)
            s += part[v][row >> 4][row & 15][c];
        if (row < a.t && n0 + c < a.n)
            a.y[(size_t)row * a.ldy + n0 + c] = s;
    }
}

template <bool XF32, bool SPLIT>
void launch_few(const ProjParams& p, hipStream_t stream)
{
    const dim3 grid((p.n + 15) / 16), block(64 * kFewWaves);
    if (p.t <= 16)
        hipLaunchKernelGGL((proj_few<1, XF32, SPLIT>), grid, block, 0, stream, p);
    else if (!XF32 || p.t <= 32)
        hipLaunchKernelGGL((proj_few<2, XF32, SPLIT>), grid, block, 0, stream, p);
    else if constexpr (XF32)
        hipLaunchKernelGGL((proj_few<4, XF32, SPLIT>), grid, block, 0, stream, p);
}

void set_tiles(ProjParams& p, uint32_t bm, uint32_t bn)
{
    p.tiles_m = (p.t + bm - 1) / bm;
    p.tiles_n = (p.n + bn - 1) / bn;
    p.tiles = p.tiles_m * p.tiles_n;
    p.per_xcd = (p.tiles + 7) / 8;
}

template <int BM, bool XF32, bool SPLIT>
void launch_proj(ProjParams p, hipStream_t stream)
{
    set_tiles(p, BM, kBN);
    hipLaunchKernelGGL((proj_tiles<BM, XF32, SPLIT>), dim3(8 * p.per_xcd), dim3(256), 0, stream, p);
}

template <int BM, int BN, int NST>
void launch_ring(ProjParams p, hipStream_t stream)
{
    set_tiles(p, BM, BN);
    hipLaunchKernelGGL((proj_ring<BM, BN, NST>), dim3(8 * p.per_xcd), dim3(256), 0, stream, p);
}

// What a call's routes are chosen by; planes: 2 with the split.
struct Size {
    uint32_t t, k, n, planes;
    bool f32;
    uint32_t cus;
};

// Workgroups in rounds over the CUs, and the share of the CUs that work in them.
struct Rounds {
    double n, share;
    Rounds(uint64_t groups, uint32_t cus) : n((double)((groups + cus - 1) / cus)), share((double)groups / (n * cus)) {}
};

// bf16 rows: the tile by an estimate of each one's time, rounds of workgroups times the time of their K stages, which
// grows with the share of the CUs that work (clock and L2), and kRoundUs a round. One round at 4096 x 4096 weights
// (64 stages), alone and on every CU: 256 x 256 78 and 109 us, 128 x 256 48 and 64, 128 x 128 28 and 36, 64 x 128 23 and
// 26, 64 x 64 18 and 19 (two rounds 36). So t = 128 takes 18 us (79 in 256 x 256 tiles), 512 26 (82), 1000 36 (83), 2048
// 64 (84), 3000 and 4096 the large tiles' 91 and 109. A tile of 128 columns must be estimated 3 % shorter than one of
// 256: about equal, the wider one was the faster (t = 3000, k = 12288, n = 4096: 256 x 256 288, 128 x 128 306).
int dma_tile(const Size& z, double& best_us)
{
    struct Tile {
        uint32_t bm, bn;
        double alone, full;  // us a stage: on an idle chip, and what a full one adds
    };
    static constexpr Tile kTiles[] = {
        {256, 256, 1.14, 0.50}, {128, 256, 0.68, 0.24}, {128, 128, 0.37, 0.12}, {64, 128, 0.28, 0.10}, {64, 64, 0.20, 0.05}};
    constexpr double kRoundUs = 3;
    int best = 0;
    for (int i = 0; i < 5; ++i) {
        const Tile& c = kTiles[i];
        const Rounds r((uint64_t)((z.t + c.bm - 1) / c.bm) * ((z.n + c.bn - 1) / c.bn), z.cus);
        const double us = r.n * (kRoundUs + z.planes * z.k / kEK * (c.alone + c.full * r.share));
        if (i == 0 || us * (c.bn < 256 && kTiles[best].bn == 256 ? 1.03 : 1) < best_us) {
            best = i;
            best_us = us;
        }
    }
    return best;
}

double rounding_us(const Size& z) { return z.f32 ? 2 + (double)z.t * z.k * (4 + 2 * z.planes) / 5e6 : 0; }

// The DMA kernels with what surrounds the tiles: the read of w and the writing of y, beside the tiles or, with the split
// (w is read twice), in part after them, and the rounding of f32 rows.
double dma_us(const Size& z)
{
    double tiles;
    dma_tile(z, tiles);
    const double bytes = 2.0 * z.k * z.n + 4.0 * z.t * z.n;
    if (z.planes == 2)
        return 1.7 + 0.91 * tiles + 0.14e-6 * bytes + rounding_us(z);
    return 1 + std::max(tiles, bytes / 4.7e6) + 0.25 * std::min(tiles, bytes / 4.7e6) + rounding_us(z);
}

// proj_few: a wave loads its share of the K chunks by U, and U past it.
double few_us(const Size& z)
{
    const uint32_t u = z.t <= 16 ? 4 : z.t <= 32 ? 2 : 1, per = kFewWaves * u;
    const double chunks = ((z.k / 64 + per - 1) / per + 1) * u, each = z.f32 ? 0.72 + 0.05 * z.t : 0.75 + 0.02 * z.t;
    const Rounds r((z.n + 15) / 16, z.cus);
    return 2.2 + r.n * chunks * each * (0.75 + 0.25 * r.share);
}

// proj_tiles: 128 rows a tile with the split, 256 without.
Rounds tiles_rounds(const Size& z)
{
    const uint32_t bm = z.planes == 2 ? 128 : 256;
    return Rounds((uint64_t)((z.t + bm - 1) / bm) * ((z.n + kBN - 1) / kBN), z.cus);
}

double tiles_us(const Size& z)
{
    const Rounds r = tiles_rounds(z);
    const double tiles = r.n * (z.planes == 2 ? 5.8 + z.k / 64 * (1.64 + 0.27 * r.share) : 8.6 + z.k / 64 * (1.75 + 0.55 * r.share));
    const double memory = (2.0 * z.k * z.n + 4.0 * z.t * z.n) / 3.9e6;
    return 1.4 + std::max(tiles, memory) + 0.12 * std::min(tiles, memory);
}

// Whether the DMA kernels take f32 rows, rounded ahead, before proj_tiles.
// With the split they read w twice, and proj_tiles, which reads it once, is the faster one where w is large and the rows
// are few, and where its tiles come out at whole rounds and K is short. us, rounded ahead / proj_tiles: t = 65, k = 4096, n
// = 4096 37 / 113, 28672 83 / 117, 65536 233 / 156; k = 2048, n = 151936 245 / 211; t = 2000, k = n = 4096 134 / 132, k =
// 512 29 / 24; t = 4096, k = n = 4096 235 / 260. Over 415 such calls (t 48 to 4096, k 64 to 14336, n 1024 to 151936) the
// estimates are within 8 % and 4 % on the average; the slower one is taken in 15, by 5 % to 14 % in seven.
// Without it they gain 3 to 15 % of a round that proj_tiles fills by more than half, the more the longer K, which must pay
// for the rounding: n = 4096, t = 4096, k = 256 24.5 / 22.1, 512 32.8 / 30.1, 1024 46.1 / 46.6. Where proj_tiles leaves
// half the chip idle, or takes several rounds, they are always faster (k = 512, t = 2000 21.5 / 28.8, n = 16384, t = 4096
// 112 / 122), and for up to 128 rows, half of its tile.
bool dma_takes(const Size& z)
{
    if (z.planes == 2)
        return dma_us(z) <= 1.02 * tiles_us(z);
    const Rounds r = tiles_rounds(z);
    return r.n > 1 || r.share <= 0.5 || z.t <= 128 || rounding_us(z) <= tiles_us(z) * (0.03 + 0.12 * z.k / 1024);
}

// Whether proj_few takes the call; `rounded`: f32 rows can be rounded ahead. Its workgroups each read all of x, so its
// time grows with n / 16 over the CUs, where the tiles' grows with the read of w: past a round or two the tiles win. us,
// w from memory, few / tiles: bf16 rows at k = 4096, t = 1: n = 4096 11.8 / 19.0, 8192 21.4 / 22.3, 16384 39 / 33, 65536
// 146 / 114; t = 32: 16.5 / 19.5, 31 / 23, 58 / 33, 225 / 116. f32 rows t = 16: 19 / 21, 37 / 25, 72 / 35, 279 / 115;
// with the split 19 / 37, 36 / 38, 69 / 51, 275 / 178. k = 14336, n = 4096, bf16 t = 32 48 / 59; k = 2048, n = 151936 312
// / 139. The estimates are within 15 % of these, the split's tiles up to a third above (the second plane's read of w comes
// in part from the last-level cache). Past kFewBf16 / F32 / Split rows the tiles win at 4096 x 4096 too (bf16
// rows 18 at 48, few 18.9; f32 20.5 at 32, few 24; split 36 at 64, few 38); without a workspace f32 rows compare with
// proj_tiles (at 4096 x 4096 122 and 114 with the split, few 38 at 64 rows).
bool few_takes(const Size& z, bool rounded)
{
    const bool dma = !z.f32 || (rounded && dma_takes(z));
    const uint32_t most = !dma ? kFewRows : !z.f32 ? kFewBf16 : z.planes == 2 ? kFewSplit : kFewF32;
    return z.t <= most && few_us(z) <= (dma ? dma_us(z) : tiles_us(z));
}

void launch_bf16(ProjParams p, uint32_t cus, hipStream_t stream)
{
    double us;
    const int best = dma_tile(Size{p.t, p.k, p.n, p.planes, false, cus}, us);
    switch (best) {
    case 0:
        set_tiles(p, kBN, kBN);
        hipLaunchKernelGGL(proj_dma, dim3(8 * p.per_xcd), dim3(256), 0, stream, p);
        break;
    case 1:
        launch_ring<128, 256, 3>(p, stream);
        break;
    case 2:
        launch_ring<128, 128, 4>(p, stream);
        break;
    case 3:
        launch_ring<64, 128, 6>(p, stream);
        break;
    default:
        launch_ring<64, 64, 8>(p, stream);
        break;
    }
}

// f32 rows are rounded into at most this much workspace.
constexpr uint64_t kMaxRounded = 256ull << 20;

// Whether a tile's DMA can address its panels by 32-bit offsets (up to 256 rows, a row's values, a margin).
bool span_fits(uint32_t rows, uint64_t ld, uint64_t k)
{
    return (uint64_t)std::min(rows, 256u) * ld * 2 + 2 * k + 128 <= 0xffffffffu;
}

bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace mako

using namespace mako;

namespace {

// (with no device the routes are the MI355X's)
Size size_of(const mako_gemm_args* a, int x_dtype, int split)
{
    const uint32_t cus = device_cus();
    return {a->t, a->k, a->n, split ? 2u : 1u, x_dtype == MAKO_F32, cus ? cus : 256u};
}

// The workspace f32 rows are rounded into (0: the call's kernels round as they load).
size_t rounded_bytes(const mako_gemm_args* a, int x_dtype, int split)
{
    const Size z = size_of(a, x_dtype, split);
    if (x_dtype != MAKO_F32 || !a->t || !a->n || !dma_takes(z) || few_takes(z, true))
        return 0;
    const uint64_t planes = split ? 2 : 1, bytes = planes * a->t * a->k * 2;
    return bytes <= kMaxRounded && span_fits(a->t, planes * a->k, planes * a->k) && span_fits(a->n, a->k, a->k) ? bytes : 0;
}

int proj_core(const mako_gemm_args* a, int x_dtype, int split, const void* w, const void* x, float* y,
              const Workspace& work, void* stream)
{
    if (!a || !w || !x || !y)
        return fail(MAKO_EINVAL, "proj: a null argument");
    if (x_dtype != MAKO_F32 && x_dtype != MAKO_BF16)
        return fail(MAKO_EUNSUPPORTED, "proj: activations of type %d (f32 or bf16)", x_dtype);
    if (a->k == 0 || a->k % 64)
        return fail(MAKO_EINVAL, "BF16 %ux%u: k must be a multiple of 64", a->k, a->n);
    if (a->row_bytes && a->row_bytes != 2 * a->k)
        return fail(MAKO_EINVAL, "proj: BF16 rows of %u values are %u bytes, not %u", a->k, 2 * a->k, a->row_bytes);
    if (split && x_dtype != MAKO_F32)
        return fail(MAKO_EINVAL, "proj: the bf16 split needs f32 activations");
    const uint32_t ldx = a->ldx ? a->ldx : a->k, ldy = a->ldy ? a->ldy : a->n;
    if (ldx < a->k || ldy < a->n)
        return fail(MAKO_EINVAL, "proj: rows of %u (x) and %u (y) are shorter than k = %u and n = %u", ldx, ldy, a->k,
                    a->n);
    if (!al16(w) || !al16(x) || ldx % 8)
        return fail(MAKO_EINVAL, "proj: w and x must be 16-byte aligned and ldx a multiple of 8");
    if ((uint64_t)a->t * ldx > 0xffffffffu || (uint64_t)a->n * a->k > 0xffffffffu)
        return fail(MAKO_EINVAL, "proj: %u x %u activations or %u x %u weights exceed 2^32 elements", a->t, ldx, a->n,
                    a->k);
    if (a->t == 0 || a->n == 0)
        return ok();
    ProjParams p{static_cast<const __bf16*>(w), x, y, a->t, a->k, a->n, ldy, ldx, 0, 0, 0, 0, 1};
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const Size z = size_of(a, x_dtype, split);
    if (x_dtype == MAKO_BF16) {
        if (!span_fits(a->t, ldx, a->k) || !span_fits(a->n, a->k, a->k))
            return fail(MAKO_EINVAL, "proj: rows of %u (x) and %u (w) values are too long for 32-bit tile offsets", ldx,
                        a->k);
        if (few_takes(z, true))
            launch_few<false, false>(p, s);
        else
            launch_bf16(p, z.cus, s);
        return check_launch("proj");
    }
    // f32 rows: rounded once into the workspace and then as bf16 rows; where it cannot be had (a capture, no memory, a
    // caller's shorter one, more than kMaxRounded bytes) the kernels round as they load.
    const uint64_t planes = split ? 2 : 1;
    const size_t bytes = rounded_bytes(a, x_dtype, split);
    if (bytes) {
        if (void* ws = work.try_get(kWsRounded, bytes, s)) {
            const dim3 grid((uint32_t)(((uint64_t)a->t * (a->k / 8) + 255) / 256));
            if (split)
                hipLaunchKernelGGL(round_rows<true>, grid, dim3(256), 0, s, static_cast<const float*>(x),
                                   static_cast<__bf16*>(ws), a->t, a->k, ldx);
            else
                hipLaunchKernelGGL(round_rows<false>, grid, dim3(256), 0, s, static_cast<const float*>(x),
                                   static_cast<__bf16*>(ws), a->t, a->k, ldx);
            p.x = ws;
            p.ldx = (uint32_t)planes * a->k;
            p.planes = (uint32_t)planes;
            launch_bf16(p, z.cus, s);
            return check_launch("proj");
        }
    }
    if (few_takes(z, false))
        split ? launch_few<true, true>(p, s) : launch_few<true, false>(p, s);
    else if (split)
        launch_proj<128, true, true>(p, s);
    else
        launch_proj<256, true, false>(p, s);
    return check_launch("proj");
}

}  // namespace

extern "C" size_t mako_proj_bf16_workspace(const mako_gemm_args* a, int x_dtype, int split)
{
    return a ? rounded_bytes(a, x_dtype, split) : 0;
}

extern "C" int mako_proj_bf16(const mako_gemm_args* a, int x_dtype, int split, const void* w, const void* x, float* y,
                              void* stream)
{
    return proj_core(a, x_dtype, split, w, x, y, library_workspace(kWsRounded, "proj"), stream);
}

extern "C" int mako_proj_bf16_ws(const mako_gemm_args* a, int x_dtype, int split, const void* w, const void* x,
                                 float* y, void* workspace, size_t workspace_bytes, void* stream)
{
    return proj_core(a, x_dtype, split, w, x, y, caller_workspace(workspace, workspace_bytes, "proj"), stream);
}
