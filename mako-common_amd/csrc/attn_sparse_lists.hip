// Block-sparse attention with one selection list per query head (sel_heads == heads: the lists cube_select writes,
// as MiniMax-H3's engine calls it, src/models/h3.cpp:357-363) for f16 heads of 128: flash_sparse_lists. The
// semantics are the reference's attention_sparse (src/kernels/ops.metal:1036-1185) as attn_sparse.hip states them:
// query tile t (64 rows) < n_cubes visits the key cubes its list names, then the dense rows [dense0, dense1); a later
// tile visits [0, n_k); keys with valid[j] == 0 are masked; causal: key j is seen by tile row r only when j <= r;
// query row r's output goes to o row map[r], dropped when map[r] < 0 or r >= n_q; lse [heads][q_pad] by tile row.
//
// Why a kernel of its own: with a list per query head, no two query tiles of a head and no two heads visit the same
// key tiles, so a staged K / V tile serves only the 64 rows of its own (head, query tile). The r64 route's sharing
// (one staged tile for the 4 waves of a workgroup) does not exist here, and a 64-rows-a-wave stream would need a ring
// of 64-key tiles per wave: more LDS than a CU holds for one wave a SIMD. So a workgroup is one (head, query tile):
// 2 waves of 32 rows over 32-key tiles, 17 KiB a tile buffer and two buffers, so that 4 workgroups (8 waves, 2 a
// SIMD) share a CU and one wave's softmax runs beside another's MFMAs.
//
// Staging is raw, by LDS DMA (16 bytes a lane, no conversion): the K image in slot order (slot s holds key
// slot_of(s), so the exponentiated scores fall in the lanes and registers of the P V B operand) with rows padded to
// 272 bytes (the 16 rows a b128 read spans start in distinct banks); the V image as the r64 stream lays it out
// (32-byte units permuted by row) and read by ds_read_b64_tr_b16 as the V^T A operand; and the tile's 32 validity
// bytes. S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16_f16, with P rounded to f16 (to nearest) as the
// reference rounds it (ops.metal:329) and the sums of the unrounded exponentials (:330); the running maximum moves
// only when a tile's passes it by more than 8 (base 2, :303-316). Tile t + 1 is in flight while tile t is computed.
// Items (head, query tile) go head-major, with every head on one XCD at a time when the heads are a multiple of 8
// (the head's K / V then stay in that XCD's L2), and the query tiles from the last (dense tiles, which see every key)
// to the first.
//
// Padding is not computed. Cubes cut by the video's edge hold few valid rows in runs of 16 (the last frame layer: one
// run of four), so a tile of 32 keys is two groups of 16 consecutive keys with a valid one, from anywhere in the
// sequence, and a workgroup's query rows are those with an output, packed. 56 heads, 9 frames of 34 x 60 patches, 948
// dense rows: 53 -> 43 thousand tiles a head, 4.33 -> 3.5 ms; one frame (16 of 64 rows valid) 901 -> 511 us with the
// selection. Without padding the list costs up to 4 % over tiles of 32 keys in a row: 16 heads, 256 cubes in lists of 32
// and 128 dense rows 612 -> 625 us, 24 heads, 100 cubes in all lists and 2000 dense rows 1128 -> 1148, 16 heads of 3000
// dense rows 106 -> 110 (a scan before the first tile), causal lists of 32 of 256 cubes 417 -> 434. (The list's next pair
// is read a tile ahead and the DMA's offsets are taken before the barrier: 642 -> 625, 1164 -> 1148 of these.) Groups of 8
// keys would save another 6 % of the first case's tiles, at four sources a tile. The loop is bound by its chain of barrier,
// scores, softmax and P V (MFMA a third busy at two waves a SIMD).
#include "fwd64_common.hpp"

namespace mako {
namespace {

constexpr uint32_t kLD = 128;                     // head dims
constexpr uint32_t kLKeys = 32;                   // keys a tile
constexpr uint32_t kLKRow = 2 * kLD + 16;         // 272: LDS bytes of a K image row
constexpr uint32_t kLKImg = 9 * 1024;             // the K image (8704 bytes) and what its ninth 1 KiB piece spills
constexpr uint32_t kLVImg = kLKeys * 2 * kLD;     // 8 KiB: the V image
constexpr uint32_t kLBuf = kLKImg + kLVImg + 64;  // and the tile's 32 validity bytes
constexpr uint32_t kLMaxSel = 256;                 // list entries a query tile
constexpr uint32_t kLGroup = 16;                  // keys a group: a tile is two groups from anywhere
constexpr uint32_t kLList = 514;                  // groups held at a time (a scan's 512 and one carried over)
constexpr float kLRescale = 8.0f;

struct ListsParams {
    const void* q;
    const void* k;
    const void* v;
    void* o;
    float* lse;
    const uint16_t* sel;
    const uint16_t* nsel;
    const uint8_t* valid;
    const int32_t* map;
    uint32_t n_q, q_pad, n_k, k_pad, heads, group, width;
    float scale_log2;
    uint32_t n_cubes, max_sel, dense0, dense1, causal, n_qt, xcd_major;
};

// An LDS DMA of 16 bytes a lane: rsrc + voff + soff to LDS m0 + 16 lane.
__device__ __forceinline__ void dma16_at(uint32_t m0, uint32_t voff, uint32_t soff, u32x4 rsrc)
{
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(m0), "v"(voff),
                 "s"(rsrc), "s"(soff)
                 : "memory", "m0");
#pragma clang diagnostic pop
}

// Where 32-byte unit u (head dims 16 u .. 16 u + 15) of V row k sits in its LDS row: u ^ (k % 4) ^ 4 (u % 2), a
// bijection of the row's 8 units for each k. A transpose read's 32-lane pass addresses units 2 db and 2 db + 1 of
// four rows k % 4 = 0 .. 3: the XOR with k % 4 spreads the rows over four units and the 4 (u % 2) term puts the odd
// unit's group in the other half of the row, so the pass covers the 64 banks once (without it, twice the 32 of one
// half: a 2-way conflict).
__device__ __forceinline__ uint32_t lv_unit(uint32_t u, uint32_t k) { return u ^ (k & 3u) ^ (4u * (u & 1u)); }
// The V byte, relative to a 1 KiB V image piece, that lane's LDS slot holds (byte 16 lane of the piece: row r,
// physical unit pu, half): the unit lv_unit places at pu, its own inverse up to the parity term.
__device__ __forceinline__ uint32_t lv_src(uint32_t lane)
{
    const uint32_t b = 16 * lane, r = b / 256, pos = b % 256, pu = pos / 32;
    const uint32_t x = pu ^ (r & 3u);
    const uint32_t u = x ^ (4u * (x & 1u));
    return r * 256 + 32 * u + 16 * ((pos / 16) & 1u);
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// x over lanes l and l ^ 32 (the two halves of a wave hold the two key halves of a row): the larger and the sum,
// both halves getting the same bits. v_permlane32_swap exchanges the upper 32 lanes of its first operand with the
// lower 32 of its second, so with x in both, one holds x of lanes 0-31 in every lane and the other x of lanes 32-63:
// no LDS round trip. The instruction goes through inline asm because this compiler's builtin returns the first
// operand for both results; the s_nop gives the preceding VALU write its wait states.
__device__ __forceinline__ void lane_halves(float x, float& lo, float& hi)
{
    uint32_t a = __builtin_bit_cast(uint32_t, x), b = a;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
    lo = __builtin_bit_cast(float, a);
    hi = __builtin_bit_cast(float, b);
}
// max(a, b, c) by one v_max3_f32: fmaxf on values the compiler cannot prove canonical (MFMA results) is a
// canonicalising v_max per operand and then the v_max, three instructions for two values.
__device__ __forceinline__ float max3(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// x where the lane's bit of the wave mask `keep` is set, -inf elsewhere: one v_cndmask on a scalar lane mask.
__device__ __forceinline__ float keep_or_ninf(float x, uint64_t keep)
{
    float r;
    asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r) : "v"(-INFINITY), "v"(x), "s"(keep));
    return r;
}

__device__ __forceinline__ float pair_max(float x)
{
    float lo, hi;
    lane_halves(x, lo, hi);
    return max3(lo, hi, -INFINITY);
}
__device__ __forceinline__ float pair_sum(float x)
{
    float lo, hi;
    lane_halves(x, lo, hi);
    return lo + hi;
}

// Four f16 of V^T by a transpose read at LDS byte `at` of this wave's group pattern.
__device__ __forceinline__ s16x4 tr_read(const unsigned char* at)
{
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at));
}

template <class TO, bool CAUSAL>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2, 2))) void flash_sparse_lists(
    const ListsParams p)
{
    using E = Elem<_Float16>;
    using V8 = f16x8;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kLBuf];
    // the groups visited, in order: K / V byte offsets (and a pair past them, read and not used)
    __shared__ __attribute__((aligned(8))) uint32_t lst[kLList + 2];
    __shared__ uint32_t lcnt[2], lcut;  // lcut: the last group crosses the end of the dense rows

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t g = lane >> 5, c32 = lane & 31;
    // The item: head-major, XCD b % 8 taking heads b % 8, b % 8 + 8, ... when xcd_major.
    uint32_t h, qt;
    {
        const uint32_t b = blockIdx.x;
        const uint32_t s = p.xcd_major ? b / 8 : b;
        h = p.xcd_major ? b % 8 + 8 * (s / p.n_qt) : s / p.n_qt;
        qt = p.n_qt - 1 - s % p.n_qt;
        if (h >= p.heads)
            return;
    }
    const uint32_t kvh = h / p.group;
    // The keys: a cube tile's selected cubes, then its dense rows; a later tile's keys [0, n_k). The list's first
    // entries, its length and the tile's row map are loaded together, Q and the first validity bytes after them: two
    // round trips before the first tile's.
    const bool cube = qt < p.n_cubes;
    const uint16_t* my_sel = p.sel + ((size_t)h * p.n_cubes + (cube ? qt : 0u)) * p.max_sel;
    const int32_t map_l = qt * 64 + lane < p.n_q ? p.map[qt * 64 + lane] : -1;
    const uint32_t sel_first = cube && tid < p.max_sel ? my_sel[tid] : 0u;
    const uint32_t ns = cube ? min(uniform_u16(p.nsel, (size_t)h * p.n_cubes + qt), p.max_sel) : 0u;
    const uint32_t dlo = cube ? p.dense0 : 0u, dhi = cube ? p.dense1 : p.n_k;
    const uint32_t nd = dhi > dlo ? (dhi - dlo + 63) / 64 : 0u;
    // The rows: those of the tile's 64 that have an output (the others, a partly filled cube's padding, are not
    // computed), packed in order, 32 a wave; a lane past the last one computes a row of zeros and stores nothing.
    uint32_t row, n_rows;
    int32_t dst;  // the row's output row
    {
        const bool has = map_l >= 0;
        const uint64_t bal = __ballot(has);
        n_rows = (uint32_t)__builtin_popcountll(bal);
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
        // lane rank of `packed` gets the lane of the rank-th such row (the others are pushed behind, in any order)
        const uint32_t at = has ? rank : n_rows + lane - rank;
        const int packed = __builtin_amdgcn_ds_permute((int)(4 * at), (int)lane);
        const int from = __builtin_amdgcn_ds_bpermute((int)(4 * (32 * w + c32)), packed);
        row = qt * 64 + (uint32_t)from;
        dst = __builtin_amdgcn_ds_bpermute(4 * from, map_l);
    }
    const bool stores = 32 * w + c32 < n_rows;
    const uint32_t row_lo = __builtin_amdgcn_readfirstlane(row);  // this wave's first row

    // Sources: the kv head's k_pad rows of K and V, the k_pad validity bytes (offsets past them load zeros).
    u32x4 krs = rsrc_of(static_cast<const _Float16*>(p.k) + (size_t)kvh * p.k_pad * kLD, p.k_pad * 2 * kLD);
    u32x4 vrs = rsrc_of(static_cast<const _Float16*>(p.v) + (size_t)kvh * p.k_pad * kLD, p.k_pad * 2 * kLD);
    u32x4 brs = rsrc_of(p.valid, p.k_pad);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        krs[i] = __builtin_amdgcn_readfirstlane(krs[i]);
        vrs[i] = __builtin_amdgcn_readfirstlane(vrs[i]);
        brs[i] = __builtin_amdgcn_readfirstlane(brs[i]);
    }
    // K image piece i (1 KiB): lane l's 16 bytes are byte 1024 i + 16 l of the image, row R = that / 272 (key
    // slot_of(R) of the tile), chunk (that % 272) / 16; chunk 16 (the row's padding) and rows past 31 (the spill of
    // piece 8) load any bytes of the tile. Wave w DMAs pieces 4 w .. 4 w + 3 and piece 8 (both waves: the same bytes
    // to the same place). V image piece i: keys 4 i .. 4 i + 3, lane l's slot holds the unit lv_unit places there.
    // slot_of keeps a row's 16, so rows 0 .. 15 come from the tile's first group and 16 .. 31 from its second: pieces
    // 0 .. 3 are the first group's, 5 .. 8 the second's, piece 4 holds row 15's end and rows 16 .. 18. Offsets are
    // within the group.
    auto kd_of = [&](uint32_t i) {
        const uint32_t b = 1024 * i + 16 * lane, r = b / kLKRow, ch = b % kLKRow / 16;
        return r < kLKeys && ch < 16 ? (slot_of(r) % kLGroup) * (2 * kLD) + 16 * ch : 0u;
    };
    uint32_t kd[5], vd[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        kd[m] = kd_of(4 * w + m);
        vd[m] = 1024 * m + lv_src(lane);
    }
    kd[4] = kd_of(8);
    const bool second = 1024 * 4 + 16 * lane >= kLGroup * kLKRow;  // piece 4's lane is the second group's
    const uint32_t lbase = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>(lds));
    // A tile's K image and validity bytes, and its V image, into buffer buf.
    // (ta, tb: the tile's groups; the wave's own is ta for wave 0 and tb for wave 1; ko: dma_k_off, taken ahead of the
    // barrier that the DMA waits for)
    auto dma_k_off = [&](uint32_t ta, uint32_t tb) __attribute__((always_inline)) {
        uint32_t ko = w == 0 ? (lane ? tb : ta) / (2 * kLD) : kd[0] + (second ? tb : ta);
        asm volatile("" : "+v"(ko));
        return ko;
    };
    auto dma_k = [&](uint32_t ta, uint32_t tb, uint32_t ko, uint32_t buf) __attribute__((always_inline)) {
        const uint32_t kb = lbase + buf * kLBuf;
        const uint32_t so = w == 0 ? ta : tb;
        dma16_at(kb + 1024 * 4 * w, w == 0 ? kd[0] : ko, w == 0 ? ta : 0u, krs);
#pragma unroll
        for (int m = 1; m < 4; ++m)
            dma16_at(kb + 1024 * (4 * w + m), kd[m], so, krs);
        dma16_at(kb + 1024 * 8, kd[4], tb, krs);
        if (w == 0 && lane < 2)
            dma16_at(kb + kLKImg + kLVImg, ko, 0, brs);
    };
    auto dma_v = [&](uint32_t ta, uint32_t tb, uint32_t buf) __attribute__((always_inline)) {
        const uint32_t vb = lbase + buf * kLBuf + kLKImg;
        const uint32_t so = w == 0 ? ta : tb;
#pragma unroll
        for (int m = 0; m < 4; ++m)
            dma16_at(vb + 1024 * (4 * w + m), vd[m], so, vrs);
    };

    // Q: the B operand, lane (c32, g) holds its row's head dims 16 kk + 8 g .. + 7 (no row: an offset past the end,
    // zeros).
    V8 qreg[8];
    {
        const auto qrs = buffer_rsrc(static_cast<const _Float16*>(p.q) + (size_t)h * p.q_pad * kLD, p.n_q * 2 * kLD);
        const uint32_t off = ((stores ? row : p.n_q) * kLD + 8 * g) * 2;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
            qreg[kk] = __builtin_bit_cast(V8, buffer_load16(qrs, off + 32 * kk));
    }
    // V^T reads: in each 16-lane group G, lane 4 j + y addresses head dims 16 (G % 2) + 4 y .. + 3 of key 8 (G / 2)
    // + j (+ 4 for the second read, + 16 for keys 16 .. 31) of 32-dim block db, and receives those dims' values for
    // four keys: unit u = 2 db + G % 2 of key row j, at lv_unit(u, j) = 4 ((db / 2) ^ (G % 2)) + ((2 (db % 2) + G % 2)
    // ^ j). Four bases, one for each db % 4; db / 4 is an immediate (none at 128 dims).
    const uint32_t gj = (lane >> 2) & 3u, gy = lane & 3u, gg = (lane >> 4) & 1u;
    uint32_t vbase[4];
#pragma unroll
    for (int d4 = 0; d4 < 4; ++d4)
        vbase[d4] = (8 * g + gj) * (2 * kLD) + 32 * lv_unit(2 * d4 + gg, gj) + 8 * gy;

    // The key sequence: the groups of 16 keys of the listed cubes, then of the dense rows, that hold a valid key (not
    // the padding of partly filled cubes) and, causal, start at or before the workgroup's last row; a tile is two
    // consecutive ones, wherever they lie. A scan finds the groups of 128 blocks of 64 keys (a cube, or 64 dense rows)
    // at once: thread i reads the 64 validity bytes of block i and the kept groups are packed in order into lst
    // (ballots, then each lane's rank); the next scan runs when the groups are used up (dense query tiles, which see
    // every key; long lists), an odd last group going to the front of the new ones.
    const uint32_t wg_last = qt * 64 + 63;
    const uint32_t n_blk = ns + nd;
    uint32_t blk = 0, used = 0, held = 0;  // the next block to scan; groups of lst taken, and held
    auto scan = [&]() __attribute__((always_inline)) {
        if (blk)
            __syncthreads();  // both waves are done with lst
        uint32_t n = 0;
        if (used < held) {
            const uint32_t carry = lst[used];
            __syncthreads();
            if (tid == 0)
                lst[0] = carry;
            n = 1;
        }
        const uint32_t i = blk + tid;
        uint32_t keep = 0, j0 = 0, hi = 0;
        if (i < n_blk) {
            const bool listed = i < ns;
            j0 = listed ? (blk ? (uint32_t)my_sel[i] : sel_first) * 64 : dlo + 64 * (i - ns);
            hi = listed ? j0 + 64 : min(dhi, j0 + 64);
            u32x4 f[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                f[k] = j0 + kLGroup * k < hi ? *reinterpret_cast<const u32x4*>(p.valid + j0 + kLGroup * k) : u32x4{};
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (((f[k][0] | f[k][1]) | (f[k][2] | f[k][3])) != 0 && (!CAUSAL || j0 + kLGroup * k <= wg_last))
                    keep |= 1u << k;
        }
        uint64_t bal[4];
        uint32_t total = 0, rank = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            bal[k] = __ballot((keep >> k) & 1u);
            total += (uint32_t)__builtin_popcountll(bal[k]);
            rank += __builtin_amdgcn_mbcnt_hi((uint32_t)(bal[k] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal[k], 0u));
        }
        if (lane == 0)
            lcnt[w] = total;
        __syncthreads();
        uint32_t at = n + (w == 1 ? lcnt[0] : 0u) + rank;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if ((keep >> k) & 1u) {
                const uint32_t j = j0 + kLGroup * k;
                lst[at++] = j * (2 * kLD);
                if (j + kLGroup > hi)
                    lcut = 1;
            }
        held = __builtin_amdgcn_readfirstlane(n + lcnt[0] + lcnt[1]);
        used = 0;
        blk += 128;
        __syncthreads();  // lst is complete
    };
    // The next tile's groups; both waves make the same calls, so they scan together. When the last tile is taken,
    // last_mask gets the keys it has (an odd tile's second group, and past the end of the dense rows, none).
    uint32_t last_mask = 0xffffffffu;
    u32x2 pair{};  // lst[used], lst[used + 1], read a tile ahead
    if (tid == 0)
        lcut = 0;
    auto next_tile = [&](uint32_t& ja, uint32_t& jb) __attribute__((always_inline)) {
        if (used + 2 >= held) {
            while (held - used < 2 && blk < n_blk) {
                scan();
                pair = *reinterpret_cast<const u32x2*>(lst);
            }
            if (used >= held)
                return false;
        }
        ja = __builtin_amdgcn_readfirstlane(pair[0]);
        jb = __builtin_amdgcn_readfirstlane(pair[1]);
        used += 2;
        pair = *reinterpret_cast<const u32x2*>(lst + used);  // (used is even)
        if (used >= held && blk >= n_blk) {
            const bool odd = used > held;
            if (odd)
                jb = ja;  // (any bytes)
            used = held;
            if (__builtin_amdgcn_readfirstlane(lcut)) {
                const uint32_t keys = (1u << (dhi - (odd ? ja : jb) / (2 * kLD))) - 1;
                last_mask = odd ? keys : keys << 16 | 0xffffu;
            } else if (odd) {
                last_mask = 0xffffu;
            }
        }
        return true;
    };

    // S^T of the tile whose K image is in buffer buf: register r holds key 8 g + r % 8 of
    // the tile's group r / 8.
    auto k_scores = [&](uint32_t buf) __attribute__((always_inline)) {
        f32x16 sc = f32x16{};
        const unsigned char* kr = lds + buf * kLBuf + c32 * kLKRow + 16 * g;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
            sc = E::mfma32(*reinterpret_cast<const V8*>(kr + 32 * kk), qreg[kk], sc);
        return sc;
    };
    // bit i: key i % 16 of group i / 16 of the tile in buffer buf is valid (last: and one of the last tile's keys)
    auto tile_mask = [&](bool last, uint32_t buf) __attribute__((always_inline)) {
        const uint32_t vflag = lds[buf * kLBuf + kLKImg + kLVImg + c32];
        const uint32_t vm = (uint32_t)__ballot(vflag != 0);
        return last ? vm & last_mask : vm;
    };
    // -inf for the scores of keys not seen: invalid, past the end of the keys or (causal) past the lane's row. Without
    // the causal limit, register r's key is a wave-uniform bit of vmask for each lane half (8 g + r % 8 + 16 (r / 8)),
    // so its lane mask is two bit tests on the scalar unit and the masking one v_cndmask a register.
    auto mask_scores = [&](f32x16& sc, uint32_t vmask, uint32_t ja, uint32_t jb) __attribute__((always_inline)) {
        if (!CAUSAL && vmask != 0xffffffffu) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int b = 16 * (r >> 3) + (r & 7);
                const uint64_t keep = (((vmask >> b) & 1u) ? 0x00000000ffffffffull : 0ull) |
                                      (((vmask >> (b + 8)) & 1u) ? 0xffffffff00000000ull : 0ull);
                sc[r] = keep_or_ninf(sc[r], keep);
            }
        } else if (CAUSAL && (vmask != 0xffffffffu || max(ja, jb) / (2 * kLD) + kLGroup - 1 > row_lo)) {
            const uint32_t lm = ((vmask >> (8 * g)) & 0xffu) | (((vmask >> (16 + 8 * g)) & 0xffu) << 8);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t j = (r < 8 ? ja : jb) / (2 * kLD) + 8 * g + (r & 7);
                sc[r] = ((lm >> r) & 1u) && j <= row ? sc[r] : -INFINITY;
            }
        }
    };

    f32x16 oacc[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
        oacc[db] = f32x16{};
    float m = -INFINITY, l = 0.0f;  // running maximum (base-2 domain) and sum of this lane's keys
    const float c = p.scale_log2;

    // Two stages: iteration t computes tile t + 1's scores (its K image, DMA'd an iteration ahead of V) beside
    // tile t's exponentials and P V. Buffer t % 2 holds K(t) and V(t); at iteration t, K(t + 2) and its validity
    // bytes go to the slot K(t) left and V(t + 1) to the slot V(t - 1) left.
    uint32_t a0 = 0, a1 = 0, b0 = 0, b1 = 0;  // the groups of tiles t and t + 1
    const bool ta = next_tile(a0, a1);
    bool tb = ta && next_tile(b0, b1);
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
        settle(qreg[kk]);
    if (ta) {
        dma_k(a0, a1, dma_k_off(a0, a1), 0);
        dma_v(a0, a1, 0);
    }
    if (tb)
        dma_k(b0, b1, dma_k_off(b0, b1), 1);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    // A wave with no row to compute (tiles of at most 32 rows with an output) stages its share of each tile and keeps
    // the barriers of the other wave's loop, then leaves.
    if (32 * w >= n_rows) {
        uint32_t bl = 0;
        for (bool have_l = ta; have_l;) {
            uint32_t c0 = 0, c1 = 0;
            const bool tc = tb && next_tile(c0, c1);
            const uint32_t ko = dma_k_off(c0, c1);
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
            if (tc)
                dma_k(c0, c1, ko, bl);
            if (tb)
                dma_v(b0, b1, bl ^ 1);
            have_l = tb;
            tb = tc;
            b0 = c0;
            b1 = c1;
            bl ^= 1;
        }
        return;
    }
    f32x16 s_cur = k_scores(0);
    mask_scores(s_cur, tile_mask(!tb, 0), a0, a1);
    uint32_t b = 0;
    bool have = ta;
    while (have) {
        uint32_t c0 = 0, c1 = 0;
        const bool tc = tb && next_tile(c0, c1);
        const uint32_t ko = dma_k_off(c0, c1);
        // this wave's DMAs of K(t + 1) and V(t) have landed; past the barrier, the other wave's too, and neither
        // reads the slots of K(t) and V(t - 1) any more
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        if (tc)
            dma_k(c0, c1, ko, b);
        if (tb)
            dma_v(b0, b1, b ^ 1);
        // tile t's row maxima and the rescale decision
        const float mx0 = max3(s_cur[0], s_cur[1], s_cur[2]), mx1 = max3(s_cur[3], s_cur[4], s_cur[5]);
        const float mx2 = max3(s_cur[6], s_cur[7], s_cur[8]), mx3 = max3(s_cur[9], s_cur[10], s_cur[11]);
        const float mx4 = max3(s_cur[12], s_cur[13], s_cur[14]);
        const float mx = pair_max(max3(max3(mx0, mx1, mx2), max3(mx3, mx4, s_cur[15]), -INFINITY)) * c;
        float f = 1.0f;
        if (mx > m + kLRescale) {
            f = exp2_fast(m - mx);
            m = mx;
        }
        l *= f;
        if (__any(f != 1.0f))
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int rr = 0; rr < 16; ++rr)
                    oacc[db][rr] *= f;
        // tile t + 1's scores (stale bytes when there is none: never used) beside tile t's exponentials
        const uint32_t vmask_n = tile_mask(!tc, b ^ 1);
        f32x16 s_nxt = k_scores(b ^ 1);
        const float mu = m == -INFINITY ? 0.0f : m;
        V8 pb[2];
        float l4[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // four chains of the row sum
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) {
            f16x8 pv;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = exp2_fast(fmaf(s_cur[8 * cc + e], c, -mu));
                l4[e & 3] += x;
                pv[e] = (_Float16)x;
            }
            pb[cc] = pv;
        }
        l += (l4[0] + l4[1]) + (l4[2] + l4[3]);
        // O^T += V^T P^T for tile t: keys 16 cc .. 16 cc + 15, head dims 32 db .. 32 db + 31.
        const unsigned char* vbuf = lds + b * kLBuf + kLKImg;
#pragma unroll
        for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                const unsigned char* va = vbuf + vbase[db] + 16 * cc * (2 * kLD);
                const s16x4 lo = tr_read(va), hi4 = tr_read(va + 4 * (2 * kLD));
                const V8 a = __builtin_bit_cast(V8, __builtin_shufflevector(lo, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
                oacc[db] = E::mfma32(a, pb[cc], oacc[db]);
            }
        mask_scores(s_nxt, vmask_n, b0, b1);
        s_cur = s_nxt;
        have = tb;
        tb = tc;
        b0 = c0;
        b1 = c1;
        b ^= 1;
    }

    // Normalise and store through the row map; the LSE by tile row.
    const float lt = pair_sum(l);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    if (stores) {
        TO* orow = static_cast<TO*>(p.o) + (size_t)dst * p.width + (size_t)h * kLD;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                store4<TO>(orow + 32 * db + 8 * r4 + 4 * g, oacc[db][4 * r4] * inv, oacc[db][4 * r4 + 1] * inv,
                           oacc[db][4 * r4 + 2] * inv, oacc[db][4 * r4 + 3] * inv);
        if (p.lse && g == 0)
            p.lse[(size_t)h * p.q_pad + row] = lt > 0.0f ? (m + __log2f(lt)) * kLn2 : -INFINITY;
    }
}

}  // namespace

// Whether a call takes flash_sparse_lists: f16 inputs, a list per query head, dense0 and k_pad multiples of 32 (so
// every tile's validity bytes lie inside valid's k_pad), valid 16-byte aligned, and the offsets in range.
bool sparse_lists_fits(const mako_sparse_args* a, mako_dtype in, const void* valid)
{
    return in == MAKO_F16 && a->kv_heads && a->heads % a->kv_heads == 0 && a->sel_heads == a->heads &&
           a->max_sel <= kLMaxSel && a->dense0 % 32 == 0 && a->k_pad % 32 == 0 &&
           (reinterpret_cast<uintptr_t>(valid) & 15u) == 0 &&
           (uint64_t)a->q_pad * 256 < (1ull << 31) && (uint64_t)a->k_pad * 256 < (1ull << 32) &&
           (uint64_t)a->heads * ((a->n_q + 63) / 64) < (1ull << 31);
}

template <class TO>
void launch_sparse_lists(const mako_sparse_args* a, float scale_log2, const void* q, const void* k, const void* v,
                         void* o, const uint16_t* sel, const uint16_t* nsel, const uint8_t* valid,
                         const int32_t* map, float* lse, hipStream_t s)
{
    const uint32_t n_qt = (a->n_q + 63) / 64;
    const ListsParams p{q,        k,          v,           o,         lse,       sel,       nsel,
                        valid,    map,        a->n_q,      a->q_pad,  a->n_k,    a->k_pad,  a->heads,
                        a->heads / a->kv_heads, a->width,  scale_log2, a->n_cubes, a->max_sel, a->dense0,
                        a->dense1, a->causal ? 1u : 0u, n_qt, a->heads % 8 == 0 ? 1u : 0u};
    if (a->causal)
        hipLaunchKernelGGL((flash_sparse_lists<TO, true>), dim3(a->heads * n_qt), dim3(128), 0, s, p);
    else
        hipLaunchKernelGGL((flash_sparse_lists<TO, false>), dim3(a->heads * n_qt), dim3(128), 0, s, p);
}

template void launch_sparse_lists<float>(const mako_sparse_args*, float, const void*, const void*, const void*,
                                         void*, const uint16_t*, const uint16_t*, const uint8_t*, const int32_t*,
                                         float*, hipStream_t);
template void launch_sparse_lists<_Float16>(const mako_sparse_args*, float, const void*, const void*, const void*,
                                            void*, const uint16_t*, const uint16_t*, const uint8_t*,
                                            const int32_t*, float*, hipStream_t);

}  // namespace mako
