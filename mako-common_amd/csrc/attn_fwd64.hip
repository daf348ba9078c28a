// Dense flash attention for heads of 128 and 64 on gfx950 with 64 query rows a wave: flash_fwd_r64.
//
// Semantics as flash_fwd (attn_fwd.hip) and the reference's flash_attn_coop (src/kernels/ops.metal:216-369): key j is
// visible to query row r (position pos = q_pos0 + r) when j < n_k && (j <= pos || (pos >= block && j >= block))
// (ops.metal:289), i.e. j < lim(pos) with lim = n_k once pos >= block and min(n_k, pos + 1) before; head h reads kv
// head h / (heads / kv_heads) (:242); the running maximum moves only when a score passes it by more than 8 in the
// base-2 domain (:303-316); P is rounded to f16 for the P V product (:329); a fully masked row gives 0 (:355); rows
// >= n_q are not stored (:359-362). The row sum adds the f32 exponentials, as the reference does (:326-331).
//
// Why this kernel beside flash_fwd: a wave of flash_fwd owns 32 rows, so each 1 KiB K / V^T operand read from LDS
// feeds one MFMA, and its vector phase and matrix phase alternate behind barriers. Here a wave owns 64 rows in two
// 32-row blocks, so each operand read feeds two MFMAs (half the LDS traffic a FLOP), one wave runs on each SIMD with
// the whole register file (O and Q in the accumulator registers, two score tiles in the vector registers), and the
// softmax of one tile runs inside the same instruction stream as the MFMAs of the next: the exponentials of tile
// j + 1 beside the P V MFMAs of tile j, the f16 packing and row sums of tile j beside the Q K^T MFMAs of tile j + 1.
// The running maximum is only recomputed when a tile's row sum shows a score above it by more than 8 (a sum over 32
// keys above 256); otherwise no maximum is formed at all. The instruction stream is generated by gen_attn_fwd64.py
// (attn_fwd64_asm.inc), which documents the schedule and the register map; this file computes the per-lane
// addresses and launches it.
//
// K / V tiles are staged through LDS as straight 16-byte copies with no conversion (LDS DMA, four buffers deep), both
// from their rows as they lie in memory: K into a padded image, V into an image whose 32-byte units are permuted by
// row, from which transpose reads (ds_read_b64_tr_b16) give the V^T operand of the P V MFMAs. P is rounded to the input
// type, so P V runs in bf16 for bf16 inputs (V exact) and in f16 for f16 inputs (the reference's rounding).
//
// A workgroup is 4 waves: hq = 4, 2 or 1 query heads of one GQA group over 256 / hq rows, so every K / V tile staged
// in LDS serves all of them. An item (a head group and a query block) is one workgroup's work; item i belongs to
// XCD i % 8, and the items of an XCD share their kv heads (causal: heaviest rows first; bidirectional: one head
// group at a time), so the K / V an XCD streams stays in its L2. The grid is persistent, one workgroup a CU, each
// walking a fixed list of its XCD's items (heavy and light in turn for causal rows), so no CU idles on the
// workgroup dispatcher between items (measured 3.5 us a handover with a grid of one workgroup an item).
#include <algorithm>
#include <type_traits>

#include "fwd64_common.hpp"

namespace mako {
namespace {

constexpr uint32_t kSplitBlocks = 128;  // query blocks a split call has at most: two a lane (SPLIT's item lookup)

struct Fwd64Params {
    const void* q;
    const void* k;
    const void* vs;   // V: its rows (flash_fwd_r64), or the V^T tile images of vt_image<T, 256> (flash_fwd_d256):
                      // [kv_heads][n_vt][256][64] f16, n_vt = ceil(n_k / 64)
    void* o;
    float* lse;
    uint32_t n_q, q_pad, n_k, k_pad, heads, kv_heads, q_pos0, block, width;
    float scale_log2;
    uint32_t group, hq, rows_wg, n_qblk, n_hg, n_vt;
    uint32_t n_items;    // n_hg x n_qblk workgroup items
};

// flash_fwd_r64's parameters with SPLIT: also tiles a piece at most; the pieces' results, po [pieces][n_q][heads][D]
// normalised f32 and pl [pieces][heads][n_q] natural-log sums; and ends[i], the pieces a head group has in its last
// i + 1 query blocks (past its n_qblk: 0xffff).
struct SplitParams : Fwd64Params {
    uint32_t piece_tiles;
    float* po;
    float* pl;
    uint16_t ends[kSplitBlocks];
};
template <bool SPLIT>
using R64Params = std::conditional_t<SPLIT, SplitParams, Fwd64Params>;

// Keys row position pos sees are [0, lim(pos)).
__device__ __forceinline__ uint32_t lim_of(uint32_t pos, uint32_t n_k, uint32_t block)
{
    return pos >= block ? n_k : min(n_k, pos + 1);
}

// The pieces an item's keys are cut into when the grid is split: np = ceil(nt / piece_tiles) nearly equal runs of
// tiles, piece i from tile start(i) up to start(i + 1). The last ones start no later than the last tile that every row
// of the item sees a key of, so no row is fully masked in the tile its piece starts with.
struct Pieces {
    uint32_t nt, np, tmax;
    __host__ __device__ Pieces(uint32_t n_tiles, uint32_t first_row_keys, uint32_t piece_tiles)
        : nt(n_tiles), np((n_tiles + piece_tiles - 1) / piece_tiles), tmax((first_row_keys - 1) / 64)
    {
    }
    __host__ __device__ uint32_t start(uint32_t i) const
    {
        const uint32_t t = i * nt / np;
        return i >= np ? nt : t < tmax ? t : tmax;
    }
};

// With SPLIT a workgroup takes pieces of items: an item's keys are cut into pieces (Pieces), a piece leaves a normalised
// f32 result and its log-sum, and merge_pieces combines them; an item of one piece is stored as without SPLIT. The
// pieces are dealt as the items are. The grid holds no idle workgroups: past one a CU the dispatcher makes a workgroup
// wait for its turn's shader engine even beside free CUs (192 pieces in a grid of 288: 35 us, alone 21).
// For calls whose items do not fill the chip or whose longest item would run on alone (split_plan).
template <class T, class TO, int D, bool SPLIT>
__global__ __launch_bounds__(256, 1) void flash_fwd_r64(const R64Params<SPLIT> p)
{
    using L = R64<D>;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[L::kLdsBytes];
    const uint32_t tid = threadIdx.x, lane = tid & 63, g = lane >> 5, c32 = lane & 31;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);

    // The grid is persistent: one workgroup a CU, each computing a fixed list of items (an item: a head group and a
    // query block), so no workgroup waits on the dispatcher between items. Item i belongs to XCD i % 8, as workgroup
    // b runs on XCD b % 8; the g8 workgroups of an XCD walk its items (x, x + 8, x + 16, ...: heaviest first for
    // causal rows) in rounds of g8, the round's order reversed every other round, so a workgroup that takes a heavy
    // item in one round takes a light one in the next. With a grid not a multiple of 8, workgroup b takes items
    // b, b + G, b + 2 G, ...
    const uint32_t G = gridDim.x, b = blockIdx.x;
    const bool by_xcd = G % 8 == 0;
    const uint32_t g8 = G / 8, bx = b % 8, bk = b / 8;
    for (uint32_t round = 0;; ++round) {
    const uint32_t item = by_xcd ? bx + 8 * (round * g8 + (round % 2 == 0 ? bk : g8 - 1 - bk)) : b + round * G;
    if (!SPLIT && item >= p.n_items)
        break;

    // Item -> (head group, query block); with SPLIT the piece too. (Braces around the unsplit form cost it 14 more spilled
    // scalar registers.)
    uint32_t hg, qb, piece = 0;
    const uint32_t id = item;
    if constexpr (SPLIT) {
        // the list of a set of `per` head groups (an XCD's, or all): blocks of rows heaviest first, for each of them
        // its pieces, for each piece the head groups
        const bool xcd_list = by_xcd && p.n_hg % 8 == 0;
        const uint32_t j = xcd_list ? item / 8 : b + round * G, per = xcd_list ? p.n_hg / 8 : p.n_hg;
        const uint16_t e0 = p.ends[lane], e1 = p.ends[lane + 64];
        const uint32_t qi = __popcll(__ballot(e0 * per <= j)) + __popcll(__ballot(e1 * per <= j));
        if (qi >= p.n_qblk)
            break;
        const uint32_t r = j - (qi ? p.ends[qi - 1] * per : 0u);
        qb = p.n_qblk - 1 - qi;
        hg = xcd_list ? bx + 8 * (r % per) : r % per;
        piece = r / per;
    } else if (p.n_hg % 8 == 0) {
        const uint32_t x = id % 8, kx = id / 8, per = p.n_hg / 8;
        if (p.block == 0) {  // bidirectional: equal work, one head group of the XCD at a time
            hg = x + 8 * (kx / p.n_qblk);
            qb = kx % p.n_qblk;
        } else {             // causal / prefix: heaviest rows first
            hg = x + 8 * (kx % per);
            qb = p.n_qblk - 1 - kx / per;
        }
    } else {
        hg = id % p.n_hg;
        qb = p.n_qblk - 1 - id / p.n_hg;
    }
    const uint32_t h = hg * p.hq + w % p.hq;
    const uint32_t kvh = hg * p.hq / p.group;
    const uint32_t wg_q0 = qb * p.rows_wg;
    const uint32_t q0 = wg_q0 + (w / p.hq) * 64;  // this wave's first row

    const uint32_t wg_last = p.q_pos0 + min(wg_q0 + p.rows_wg, p.n_q) - 1;
    uint32_t n_keys = wg_last >= p.block ? p.n_k : min(p.n_k, wg_last + 1);
    // the piece's first key: limits and counts below are relative to it
    uint32_t ks = 0;
    bool partial = false;
    if constexpr (SPLIT) {
        const Pieces pc((n_keys + 63) / 64, lim_of(p.q_pos0 + wg_q0, p.n_k, p.block), p.piece_tiles);
        if (pc.start(piece) >= pc.start(piece + 1))
            continue;  // an empty piece (prefix-causal rows: most of the keys lie past the first row's)
        partial = pc.np > 1;
        ks = 64 * pc.start(piece);
        n_keys = min(n_keys, 64 * pc.start(piece + 1)) - ks;
    }
    const bool live = q0 < p.n_q;
    const uint32_t w_last = p.q_pos0 + min(q0 + 64, p.n_q) - 1;
    const uint32_t w_lim = !live ? 0u : (w_last >= p.block ? p.n_k : min(p.n_k, w_last + 1));
    const uint32_t w_keys = SPLIT && live ? min(n_keys, w_lim - ks) : w_lim;
    const uint32_t nt = (n_keys + 63) / 64, ntw = (w_keys + 63) / 64;
    const uint32_t p0 = p.q_pos0 + q0;
    const uint32_t lmin = lim_of(p0, p.n_k, p.block) - ks;
    const uint32_t lim0 = lim_of(p0 + c32, p.n_k, p.block) - ks - 8 * g;
    const uint32_t lim1 = lim_of(p0 + 32 + c32, p.n_k, p.block) - ks - 8 * g;

    // LDS: the K images, then the V images.
    const uint32_t lbase = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    const uint32_t vbase = lbase + kNBuf * L::kKTile;
    uint32_t kr = lbase + c32 * L::kKRow + 16 * g;  // K fragment reads (buffer 0)
    const uint32_t kr0 = kr;
    // V transpose reads (buffer 0): lane 32 g + 16 h + i addresses row 8 g + i / 4 of a fragment's keys, bytes
    // 8 (i % 4) of its unit 2 db + h, which sits at v_unit(2 db + h, i / 4); vr0 for even db, vr1 for odd.
    const uint32_t th = (lane >> 4) & 1u, ti = lane & 15u;
    const uint32_t vrow = vbase + (8 * g + ti / 4) * L::kVRow + 8 * (ti % 4);
    uint32_t vr0 = vrow + 32 * v_unit(th, ti / 4);
    uint32_t vr1 = vrow + 32 * v_unit(2 + th, ti / 4);
    // Staging. K image piece i (bytes 1024 i .. + 1023 of the padded tile): lane l holds byte b = 1024 i + 16 l, row
    // R = b / kKRow (the row of key slot_of(R)), chunk b % kKRow / 16 (chunk D / 8 is the row's padding: any bytes
    // of the row will do). The wave stages pieces w + 4 m (m < kNKP: 4 at D 128, 2 at D 64) and the last piece,
    // 4 kNKP. V: the wave's quarter of the image (4 or 2 KiB, rows 16 w ..), vd_of(lane) from each piece's start.
    auto kd_of = [&](uint32_t i) {
        const uint32_t b = 1024 * i + 16 * lane, row = b / L::kKRow, ch = b % L::kKRow / 16;
        return slot_of(row) * (2 * D) + 16 * (ch < D / 8 ? ch : 0);
    };
    const uint32_t kd0 = kd_of(w), kd1 = kd_of(w + 4);
    const uint32_t kd2 = L::kNKP > 2 ? kd_of(w + 8) : 0u, kd3 = L::kNKP > 3 ? kd_of(w + 12) : 0u;
    const uint32_t kd4 = kd_of(4 * L::kNKP);
    const uint32_t vd = (L::kVTile / 4) * w + vd_of<D>(lane);
    // LDS DMA destinations (buffer 0): K image, this wave's first K piece, its 4 KiB of the V image
    const uint32_t skw = __builtin_amdgcn_readfirstlane(lbase), skww = __builtin_amdgcn_readfirstlane(lbase + 1024 * w);
    const uint32_t svww = __builtin_amdgcn_readfirstlane(vbase + (L::kVTile / 4) * w);
    const uint32_t qo = ((q0 + c32) * D + 8 * g) * 2;
    // Epilogue: the wave's rows of O go through its own LDS region (64 rows of D * so bytes, 16-byte chunk c of
    // row R at c ^ (R % 8)). ew: where the lane's pieces of row c32 go (with the lane's part of the chunk index and
    // the swizzle; the stream xors in the rest); er: the first whole-row chunk it reads back (lane l: row l / lpr,
    // chunk l % lpr, lpr = lanes a row); og: where that chunk goes in o; ogs: o bytes of one read's rows.
    const uint32_t so = SPLIT && partial ? 4u : (uint32_t)sizeof(TO), orow = D * so, lpr = orow / 16;
    const uint32_t width = SPLIT && partial ? p.heads * D : p.width;
    const uint32_t obase = lbase + w * 64 * orow;
    const uint32_t ew = so == 4 ? obase + c32 * orow + 16 * ((c32 & 7u) ^ g)
                                : obase + c32 * orow + 8 * g + 16 * (c32 & 7u);
    const uint32_t er = obase + (lane / lpr) * orow + 16 * ((lane % lpr) ^ (lane / lpr));
    const uint32_t og = (q0 + lane / lpr) * width * so + h * orow + 16 * (lane % lpr);
    const uint32_t ogs = __builtin_amdgcn_readfirstlane((64 / lpr) * width * so);
    const uint32_t lo0 = q0 + c32 < p.n_q ? (h * p.n_q + q0 + c32) * 4 : 0xffffffffu;
    const uint32_t lo1 = q0 + 32 + c32 < p.n_q ? (h * p.n_q + q0 + 32 + c32) * 4 : 0xffffffffu;
    const uint32_t swp = (lane ^ 32) * 4;

    const u32x4 qrs = rsrc_of(static_cast<const T*>(p.q) + (size_t)h * p.q_pad * D, p.n_q * 2 * D);
    const u32x4 krs = rsrc_of(static_cast<const T*>(p.k) + ((size_t)kvh * p.k_pad + ks) * D, n_keys * 2 * D);
    const u32x4 vrs = rsrc_of(static_cast<const T*>(p.vs) + ((size_t)kvh * p.k_pad + ks) * D, n_keys * 2 * D);
    void* out = p.o;
    float* lse = p.lse;
    if constexpr (SPLIT) {
        if (partial) {
            out = p.po + (size_t)piece * p.n_q * width;
            lse = p.pl + (size_t)piece * p.heads * p.n_q;
        }
    }
    const u32x4 ors = rsrc_of(out, p.n_q * width * so);
    const u32x4 lrs = rsrc_of(lse, lse ? p.heads * p.n_q * 4 : 0);
    // scalar operands, made wave-uniform explicitly (the asm reads them from scalar registers)
    const uint32_t has_lse = __builtin_amdgcn_readfirstlane(lse ? 1u : 0u);
    const float c = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(uint32_t, p.scale_log2)));
    const uint32_t s_nt = __builtin_amdgcn_readfirstlane(nt), s_ntw = __builtin_amdgcn_readfirstlane(ntw);
    const uint32_t s_lmin = __builtin_amdgcn_readfirstlane(lmin);
    const uint32_t kb0 = __builtin_amdgcn_readfirstlane(krs[0]), kb1 = __builtin_amdgcn_readfirstlane(krs[1]);
    const uint32_t kn = __builtin_amdgcn_readfirstlane(krs[2]);
    const uint32_t vb0 = __builtin_amdgcn_readfirstlane(vrs[0]), vb1 = __builtin_amdgcn_readfirstlane(vrs[1]);
    const uint32_t vn = __builtin_amdgcn_readfirstlane(vrs[2]);

#define MAKO_FWD64_OPERANDS                                                                                     \
    : [kr] "+v"(kr), [vr0] "+v"(vr0), [vr1] "+v"(vr1)                                                           \
    : [kd0] "v"(kd0), [kd1] "v"(kd1), [kd2] "v"(kd2), [kd3] "v"(kd3), [kd4] "v"(kd4), [vd] "v"(vd),              \
      [lim0] "v"(lim0), [lim1] "v"(lim1), [kr0] "v"(kr0), [qo] "v"(qo), [lo0] "v"(lo0), [lo1] "v"(lo1),          \
      [swp] "v"(swp), [ew] "v"(ew), [er] "v"(er), [og] "v"(og), [qrs] "s"(qrs), [ors] "s"(ors), [lrs] "s"(lrs),    \
      [c] "s"(c), [nt] "s"(s_nt), [ntw] "s"(s_ntw), [lmin] "s"(s_lmin), [has_lse] "s"(has_lse), [ogs] "s"(ogs),    \
      [kb0] "s"(kb0),                                                                                             \
      [kb1] "s"(kb1), [kn] "s"(kn), [vb0] "s"(vb0), [vb1] "s"(vb1), [vn] "s"(vn), [skw] "s"(skw),               \
      [skww] "s"(skww), [svww] "s"(svww)                                                                          \
    : MAKO_FWD64_CLOBBERS, "vcc", "scc", "memory"

#define MAKO_FWD64_STREAM(NAME, OUT16)                                                                            \
    do {                                                                                                        \
        if (__is_same(TO, float) || (SPLIT && partial))                                                         \
            asm volatile(NAME##_F32 MAKO_FWD64_OPERANDS);                                                       \
        else                                                                                                    \
            asm volatile(NAME##_##OUT16 MAKO_FWD64_OPERANDS);                                                   \
    } while (0)

    if constexpr (D == 64) {
        if constexpr (__is_same(T, __bf16))
            MAKO_FWD64_STREAM(MAKO_FWD64_D64_ASM_BF16, BF16);
        else
            MAKO_FWD64_STREAM(MAKO_FWD64_D64_ASM_F16, F16);
    } else if constexpr (__is_same(T, __bf16)) {
        MAKO_FWD64_STREAM(MAKO_FWD64_ASM_BF16, BF16);
    } else {
        MAKO_FWD64_STREAM(MAKO_FWD64_ASM_F16, F16);
    }
    // every wave's stream has ended (its LDS reads landed) before the next item's staging overwrites LDS
    asm volatile("s_barrier" ::: "memory");
    }
#undef MAKO_FWD64_STREAM
#undef MAKO_FWD64_OPERANDS
}

// The rows of items with more than one piece, from query row row0 on: the pieces' normalised rows weighted by
// exp(their log-sum - the largest). D / 4 lanes a (row, head), four head dims each; bound by the read of the pieces.
// A piece whose sum is not above 0 has a log-sum of -inf: zeros where every score was -inf, NaN where one was not a
// number. Its row is added with weight 0, so NaN reaches the result whichever piece it is in; a row that is NaN
// throughout makes the sum NaN too, and so the log-sum -inf, as in the call without pieces.
template <class TO, int D>
__global__ __launch_bounds__(256) void merge_pieces(const SplitParams p, uint32_t row0)
{
    const uint32_t t = blockIdx.x * (1024 / D) + threadIdx.x / (D / 4), d = 4 * (threadIdx.x % (D / 4));
    const uint32_t row = row0 + t / p.heads, h = t % p.heads;
    if (row >= p.n_q)
        return;
    const uint32_t wg_q0 = row / p.rows_wg * p.rows_wg, last = p.q_pos0 + min(wg_q0 + p.rows_wg, p.n_q) - 1;
    const Pieces pc((lim_of(last, p.n_k, p.block) + 63) / 64, lim_of(p.q_pos0 + wg_q0, p.n_k, p.block), p.piece_tiles);
    const float* pl = p.pl + (size_t)h * p.n_q + row;
    const float* po = p.po + ((size_t)row * p.heads + h) * D + d;
    const size_t ls = (size_t)p.heads * p.n_q, os = ls * D;
    constexpr uint32_t U = 4;  // pieces whose loads are in flight together
    float mx = -INFINITY, sum = 0.0f;
    f32x4 acc = f32x4{};
    for (uint32_t i0 = 0; i0 < pc.np; i0 += U) {
        float l[U];
        f32x4 v[U];
        #pragma unroll
        for (uint32_t u = 0; u < U; ++u) {  // (an empty piece wrote nothing: zeros)
            const bool has = i0 + u < pc.np && pc.start(i0 + u) < pc.start(i0 + u + 1);
            l[u] = has ? pl[(i0 + u) * ls] : -INFINITY;
            v[u] = has ? *reinterpret_cast<const f32x4*>(po + (i0 + u) * os) : f32x4{};
        }
        #pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            if (l[u] == -INFINITY) {  // (the same in a row's lanes)
                const uint64_t nan = __ballot(v[u][0] != v[u][0] && v[u][1] != v[u][1] && v[u][2] != v[u][2] && v[u][3] != v[u][3]);
                const uint64_t row_lanes = ((1ull << (D / 4)) - 1) << (threadIdx.x & 63u & ~(D / 4 - 1));
                acc += v[u] * 0.0f;
                if ((nan & row_lanes) == row_lanes)
                    sum = NAN;
                continue;
            }
            const float m = fmaxf(mx, l[u]);
            const float a = exp2_fast((mx - m) * kLog2e), b = exp2_fast((l[u] - m) * kLog2e);
            sum = sum * a + b;
            acc = acc * a + v[u] * b;
            mx = m;
        }
    }
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
    store4<TO>(static_cast<TO*>(p.o) + (size_t)row * p.width + (size_t)h * D + d, acc[0] * inv, acc[1] * inv,
               acc[2] * inv, acc[3] * inv);
    if (p.lse && d == 0)
        p.lse[(size_t)h * p.n_q + row] = sum > 0.0f ? mx + __log2f(sum) * kLn2 : -INFINITY;
}

// Heads of 256 (Qwen3.5's gated attention): flash_fwd_d256. The parallelism of the usual shapes (16 query heads,
// causal) needs items of 32 rows a wave, and a 256-wide O of 32 rows is 128 accumulator registers, so this kernel
// keeps flash_fwd_wide's shape: 4 waves, one a SIMD, hq heads x 128 / hq rows a workgroup, two 64-key tile buffers,
// S^T = K Q^T and O^T += V^T P^T on 32x32x16 MFMAs with Q in registers. What it changes is the staging: K as the
// padded image (rows of 528 bytes, slot order) and V^T from the f16 tile images of vt_image<T, 256>, both by LDS DMA,
// 16 bytes a lane with no conversion, so the transposes, conversions and LDS writes that took most of the vector
// instructions of flash_fwd_wide's loop are gone from it. A tile's 33 KiB of K image and 32 KiB of V^T: wave w DMAs
// K pieces w + 4 m (m < 8) and piece 32 (every wave; the same bytes to the same place), and its 8 KiB of V^T.
// Tile jb + 1 is in flight while tile jb is computed; each iteration ends with this wave's DMAs landed and the
// workgroup barrier (the buffer just read is then free, the next one full).
__device__ __forceinline__ void dma16(uint32_t m0, uint32_t voff, u32x4 rsrc)
{
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(m0), "v"(voff),
                 "s"(rsrc)
                 : "memory", "m0");
#pragma clang diagnostic pop
}

template <class T, class TO>
__global__ __launch_bounds__(256, 1) void flash_fwd_d256(const Fwd64Params p)
{
    constexpr int D = 256;
    using L = R64<D>;
    using E = Elem<T>;
    using V8 = typename E::vec8;
    using H = Elem<_Float16>;
    using H8 = f16x8;
    constexpr int NDB = D / 32, NKK = D / 16;
    constexpr uint32_t kBuf = L::kKTile + L::kVTile;  // 33 + 32 KiB
    __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kBuf];

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t g = lane >> 5, c32 = lane & 31;
    const uint32_t hg = blockIdx.x;
    const uint32_t qb = p.n_qblk - 1 - blockIdx.y;  // the latest rows (the most keys) first
    const uint32_t h = hg * p.hq + w % p.hq;
    const uint32_t kvh = hg * p.hq / p.group;
    const uint32_t wg_q0 = qb * p.rows_wg;
    const uint32_t q0 = wg_q0 + (w / p.hq) * 32;  // this wave's first row

    // Keys the workgroup visits (the causal bound), and this wave's own bound.
    const uint32_t wg_last = p.q_pos0 + min(wg_q0 + p.rows_wg, p.n_q) - 1;
    const uint32_t n_keys = wg_last >= p.block ? p.n_k : min(p.n_k, wg_last + 1);
    const bool live = q0 < p.n_q;
    const uint32_t w_last = p.q_pos0 + min(q0 + 32, p.n_q) - 1;
    const uint32_t w_keys = !live ? 0u : (w_last >= p.block ? p.n_k : min(p.n_k, w_last + 1));
    const uint32_t p0 = p.q_pos0 + q0;
    const uint32_t pos = p0 + c32;

    // Sources: K rows of this kv head up to n_keys (rows past it load as zeros), its V^T tile images.
    const uint32_t nb = (n_keys + 63) / 64;
    u32x4 krs = rsrc_of(static_cast<const T*>(p.k) + (size_t)kvh * p.k_pad * D, n_keys * 2 * D);
    u32x4 vrs = rsrc_of(static_cast<const unsigned char*>(p.vs) + (size_t)kvh * p.n_vt * L::kVTile,
                        p.n_vt * L::kVTile);
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
        krs[i] = __builtin_amdgcn_readfirstlane(krs[i]);
        vrs[i] = __builtin_amdgcn_readfirstlane(vrs[i]);
    }
    // K image piece i: lane l's 16 bytes are byte 1024 i + 16 l of the padded tile: row R = that / 528 (key
    // slot_of(R) of the tile), chunk (that % 528) / 16 (chunk 32 is the row's padding: any bytes of it will do).
    auto kd_of = [&](uint32_t i) {
        const uint32_t b = 1024 * i + 16 * lane, row = b / L::kKRow, ch = b % L::kKRow / 16;
        return slot_of(row) * (2 * D) + 16 * (ch < D / 8 ? ch : 0);
    };
    uint32_t kd[9];
    #pragma unroll
    for (int m = 0; m < 8; ++m)
        kd[m] = kd_of(w + 4 * m);
    kd[8] = kd_of(32);
    const uint32_t lbase = __builtin_amdgcn_readfirstlane((uint32_t)reinterpret_cast<uintptr_t>(lds));
    // DMA instruction i (0 .. 16) of this wave's share of tile t into buffer buf: K pieces (i < 9), then V^T
    auto dma_piece = [&](uint32_t t, uint32_t buf, int i) __attribute__((always_inline)) {
        const uint32_t kb = lbase + buf * kBuf, vb = kb + L::kKTile;
        if (i < 8)
            dma16(kb + 1024 * (w + 4 * i), t * (64 * 2 * D) + kd[i], krs);
        else if (i == 8)
            dma16(kb + 1024 * 32, t * (64 * 2 * D) + kd[8], krs);
        else
            dma16(vb + (L::kVTile / 4) * w + 1024 * (i - 9),
                  t * L::kVTile + (L::kVTile / 4) * w + 16 * lane + 1024 * (i - 9), vrs);
    };
    auto dma_tile = [&](uint32_t t, uint32_t buf) __attribute__((always_inline)) {
        #pragma unroll
        for (int i = 0; i < 17; ++i)
            dma_piece(t, buf, i);
    };

    // Q: the B operand, lane (c32, g) holds row q0 + c32, head dims 16 kk + 8 g .. + 7 (rows past n_q load as 0).
    V8 qreg[NKK];
    {
        const auto qrs = buffer_rsrc(static_cast<const T*>(p.q) + (size_t)h * p.q_pad * D, p.n_q * D * sizeof(T));
        const uint32_t off = ((q0 + c32) * D + 8 * g) * sizeof(T);
        #pragma unroll
        for (int kk = 0; kk < NKK; ++kk)
            qreg[kk] = __builtin_bit_cast(V8, buffer_load16(qrs, off + 16 * kk * sizeof(T)));
        #pragma unroll
        for (int kk = 0; kk < NKK; ++kk)
            settle(qreg[kk]);
    }

    f32x16 oacc[NDB];
    #pragma unroll
    for (int db = 0; db < NDB; ++db)
        oacc[db] = f32x16{};
    float m = -INFINITY, l = 0.0f;  // running maximum (base-2 domain) and sum of this lane's keys
    const float c = p.scale_log2;
    const uint32_t sw = vt_swz(c32);  // the V^T rows this lane reads are 32 db + c32: the swizzle of c32

    if (nb > 0)
        dma_tile(0, 0);
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    // Tile jb's exponentials against the running maximum, P V, and the barrier that ends the iteration.
    f32x16 s[2];
    auto finish_tile = [&](uint32_t jb) __attribute__((always_inline)) {
        const uint32_t buf = jb & 1;
        if (jb * 64 < w_keys) {
            const unsigned char* vbuf = lds + buf * kBuf + L::kKTile;
            const float mu = m == -INFINITY ? 0.0f : m;
            // P in f16 as the B operand of O^T += V^T P^T: chunk 2 t + a holds keys j0 + 32 t + 16 a + 8 g + 0..7.
            // Chunk cc + 1's exponentials run beside chunk cc's MFMAs, one key a slot, and the V^T fragments are
            // read three MFMAs ahead of their use (a ring of four), in the order the MFMAs take them.
            H8 pb[4];
            u32x4 pk[4];
            float ev[4][4];  // the even key of each pair until its odd one is packed beside it
            auto key = [&](int cc, int e) __attribute__((always_inline)) {  // key e (0 .. 7) of chunk cc
                const int t = cc / 2, a = cc % 2;
                const float x = exp2_fast(fmaf(s[t][8 * a + e], c, -mu));
                l += x;
                if (e % 2 == 0)
                    ev[cc][e / 2] = x;
                else
                    pk[cc][e / 2] = H::pack2(ev[cc][e / 2], x);
            };
            // V^T rows 32 db + c32 of the image: 128 bytes a row, keys 8 s' .. + 7 in 16-byte slot s' ^ vt_swz(row).
            H8 vf[4];
            auto vread = [&](int i) __attribute__((always_inline)) {  // the fragment of MFMA i = 8 cc + db
                const int cc = i / NDB, db = i % NDB;
                const unsigned char* vr = vbuf + c32 * 128 + 16 * (((2 * cc + g) ^ sw) & 7u);
                vf[i % 4] = *reinterpret_cast<const H8*>(vr + 4096 * db);
            };
            vread(0);
            vread(1);
            vread(2);
            #pragma unroll
            for (int e = 0; e < 8; ++e)
                key(0, e);
            pb[0] = __builtin_bit_cast(H8, pk[0]);
            __builtin_amdgcn_sched_barrier(0);
            #pragma unroll
            for (int i = 0; i < 4 * NDB; ++i) {
                const int cc = i / NDB, db = i % NDB;
                if (i + 3 < 4 * NDB)
                    vread(i + 3);
                __builtin_amdgcn_sched_barrier(0);
                if (cc + 1 < 4)
                    key(cc + 1, db);
                oacc[db] = H::mfma32(vf[i % 4], pb[cc], oacc[db]);
                if (db == NDB - 1 && cc + 1 < 4)
                    pb[cc + 1] = __builtin_bit_cast(H8, pk[cc + 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // this wave's DMAs of tile jb + 1 have landed and every wave is done with buffer buf
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };

    // The loop over tiles carries no vector work on the accumulators: when a tile's maximum moves the running one
    // (rarely: by more than 8, base 2), control leaves the inner loop, and the rescale of O and that tile's P V run
    // outside it. Inside it, the compiler would keep a second copy of O in vector registers for the rescale, made
    // anew every tile.
    uint32_t jb = 0;
    float mx = -INFINITY;
    for (;;) {
        bool moved = false;
        for (; jb < nb; ++jb) {
            const uint32_t buf = jb & 1;
            const uint32_t j0 = jb * 64;
            const bool next = jb + 1 < nb;  // tile jb + 1 goes to buffer buf ^ 1 (read last in tile jb - 1)
            if (next && j0 >= w_keys)
                dma_tile(jb + 1, buf ^ 1);
            if (j0 < w_keys) {
                const unsigned char* kbuf = lds + buf * kBuf;
                // S^T for keys j0 .. j0 + 63: register r of tile t holds key j0 + 32 t + 16 (r / 8) + 8 g + r % 8.
                s[0] = f32x16{};
                s[1] = f32x16{};
                {
                    // K fragments read two K steps ahead of their MFMAs (a ring of three pairs)
                    const unsigned char* kr0 = kbuf + c32 * L::kKRow + 16 * g;
                    const unsigned char* kr1 = kr0 + 32 * L::kKRow;
                    V8 kf[3][2];
                    auto kread = [&](int kk) __attribute__((always_inline)) {
                        kf[kk % 3][0] = *reinterpret_cast<const V8*>(kr0 + 32 * kk);
                        kf[kk % 3][1] = *reinterpret_cast<const V8*>(kr1 + 32 * kk);
                    };
                    kread(0);
                    kread(1);
                    __builtin_amdgcn_sched_barrier(0);
                    // the next tile's 17 DMA instructions go out one beside each score MFMA pair (the last two
                    // together), so no MFMA waits behind their issue; one branch chooses the form
                    auto scores = [&](auto DMA) __attribute__((always_inline)) {
                        #pragma unroll
                        for (int kk = 0; kk < NKK; ++kk) {
                            if (kk + 2 < NKK)
                                kread(kk + 2);
                            __builtin_amdgcn_sched_barrier(0);
                            s[0] = E::mfma32(kf[kk % 3][0], qreg[kk], s[0]);
                            if constexpr (decltype(DMA)::value)
                                dma_piece(jb + 1, buf ^ 1, kk);
                            s[1] = E::mfma32(kf[kk % 3][1], qreg[kk], s[1]);
                            if constexpr (decltype(DMA)::value)
                                if (kk == NKK - 1)
                                    dma_piece(jb + 1, buf ^ 1, 16);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    };
                    if (next)
                        scores(std::true_type{});
                    else
                        scores(std::false_type{});
                }
                const bool plain = j0 + 64 <= p.n_k && (j0 + 63 <= p0 || (p0 >= p.block && j0 >= p.block));
                if (!plain) {
                    const bool lane_open = pos >= p.block;
                    #pragma unroll
                    for (int t = 0; t < 2; ++t)
                        #pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const uint32_t j = j0 + 32 * t + 16 * (r >> 3) + 8 * g + (r & 7);
                            const bool seen = (j < p.n_k) & ((j <= pos) | (lane_open & (j >= p.block)));
                            s[t][r] = seen ? s[t][r] : -INFINITY;
                        }
                }
                mx = -INFINITY;
                #pragma unroll
                for (int t = 0; t < 2; ++t)
                    #pragma unroll
                    for (int r = 0; r < 16; ++r)
                        mx = fmaxf(mx, s[t][r]);
                mx = fmaxf(mx, swap_halves(mx)) * c;  // the row's maximum, base 2 (c > 0)
                if (__any(mx > m + 8.0f)) {
                    moved = true;
                    break;
                }
            }
            finish_tile(jb);
        }
        if (!moved)
            break;
        // the rescale: rows whose maximum passed theirs by more than 8 move it (f = 0 while nothing was seen)
        float f = 1.0f;
        if (mx > m + 8.0f) {
            f = exp2_fast(m - mx);
            m = mx;
        }
        l *= f;
        #pragma unroll
        for (int db = 0; db < NDB; ++db)
            #pragma unroll
            for (int r = 0; r < 16; ++r)
                oacc[db][r] *= f;
        finish_tile(jb);
        ++jb;
    }

    // The row's sum over both halves of the wave; normalise. Register r of output block db holds head dim 32 db +
    // 8 (r / 4) + 4 g + r % 4 of row q0 + c32. O goes through LDS (free: the loop's last barrier is behind every
    // wave's reads): each wave writes its 32 rows into its own region, row-major with 16-byte chunk ch of row R at
    // ch ^ R, then reads back whole chunks of whole rows, so each global store covers contiguous row segments (1 KiB
    // an instruction) instead of 8 or 16 bytes of each of 32 rows.
    const float lt = l + swap_halves(l);
    const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
    const uint32_t row = q0 + c32;
    if (live && row < p.n_q && p.lse && g == 0)
        p.lse[(size_t)h * p.n_q + row] = lt > 0.0f ? (m + __log2f(lt)) * kLn2 : -INFINITY;
    constexpr uint32_t kRowB = D * sizeof(TO);  // bytes of an O row: 512 (16-bit) or 1024 (f32)
    unsigned char* orgn = lds + w * 32 * kRowB;
    #pragma unroll
    for (int db = 0; db < NDB; ++db)
        #pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const uint32_t byte = (32 * db + 8 * r4 + 4 * g) * sizeof(TO);
            TO* at = reinterpret_cast<TO*>(orgn + c32 * kRowB + 16 * ((byte / 16) ^ c32) + byte % 16);
            store4<TO>(at, oacc[db][4 * r4] * inv, oacc[db][4 * r4 + 1] * inv, oacc[db][4 * r4 + 2] * inv,
                       oacc[db][4 * r4 + 3] * inv);
        }
    if (live) {
        unsigned char* obase = static_cast<unsigned char*>(p.o) + ((size_t)q0 * p.width + (size_t)h * D) * sizeof(TO);
        #pragma unroll
        for (uint32_t i = 0; i < 32 * kRowB / 1024; ++i) {
            const uint32_t flat = 1024 * i + 16 * lane, r = flat / kRowB, ch = flat % kRowB / 16;
            const u32x4 x = *reinterpret_cast<const u32x4*>(orgn + r * kRowB + 16 * (ch ^ r));
            if (q0 + r < p.n_q)
                __builtin_nontemporal_store(x, reinterpret_cast<u32x4*>(obase + (size_t)r * p.width * sizeof(TO) +
                                                                         16 * ch));
        }
    }
}

}  // namespace

// Whether flash_fwd_r64 for heads of D takes the call: its sizes fit the kernel's 32-bit buffer offsets.
template <int D>
bool fwd64_fits(const mako_attn_args* a, uint32_t out_bytes)
{
    using L = R64<D>;
    const uint32_t group = a->heads / a->kv_heads;
    const uint32_t hq = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const uint32_t rows_wg = 256 / hq;
    const uint64_t o_rows = (uint64_t)((a->n_q + rows_wg - 1) / rows_wg) * rows_wg + 64;
    return o_rows * a->width * out_bytes < (1ull << 32) && (uint64_t)a->heads * a->n_q * 4 < (1ull << 32) &&
           (uint64_t)a->k_pad * 2 * D + 4 * L::kVTile < (1ull << 32) && (uint64_t)a->q_pad * 2 * D < (1ull << 31);
}
template bool fwd64_fits<128>(const mako_attn_args*, uint32_t);
template bool fwd64_fits<64>(const mako_attn_args*, uint32_t);

// Whether flash_fwd_d256 takes the call (32-bit offsets, the grid).
bool d256_fits(const mako_attn_args* a)
{
    using L = R64<256>;
    const uint32_t group = a->heads / a->kv_heads;
    const uint32_t hq = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const uint32_t n_qblk = (a->n_q + 128 / hq - 1) / (128 / hq);
    const uint32_t n_vt = (a->n_k + 63) / 64;
    return (uint64_t)a->k_pad * 512 + 2 * L::kKTile < (1ull << 32) && (uint64_t)n_vt * L::kVTile < (1ull << 32) &&
           (uint64_t)a->q_pad * 512 < (1ull << 31) && n_qblk <= 65535;
}

namespace {

// How a call's keys are split over workgroups (pieces 1: they are not).
struct SplitPlan {
    uint32_t piece_tiles = 0, pieces = 1;
    uint32_t row0 = 0;  // the first query row of an item with more than one piece
    size_t o_bytes = 0, bytes = 0;
};

// The 64-key tiles the items of query block qb walk.
uint32_t item_tiles(const mako_attn_args* a, uint32_t rows_wg, uint32_t qb)
{
    const uint32_t last = a->q_pos0 + std::min((qb + 1) * rows_wg, a->n_q) - 1;
    return ((last >= a->block ? a->n_k : std::min(a->n_k, last + 1)) + 63) / 64;
}

// The keys query row `row` sees.
uint32_t first_keys(const mako_attn_args* a, uint32_t row)
{
    const uint32_t pos = a->q_pos0 + row;
    return pos >= a->block ? a->n_k : std::min(a->n_k, pos + 1);
}

// An estimate in microseconds, from this kernel's times: a workgroup takes kTileUs a tile of 64 keys on an otherwise
// idle chip and kFullUs more where every CU works (the clock drops), kWgUs around them (dispatch, prologue, epilogue)
// and kTurnUs for each further piece; the merge kMergeUs and its read of the pieces. A plan must gain 15 %.
// Measured at 32 / 8 heads of 128, unsplit and split: 333 rows over 9333 keys 174 -> 61 us, 100 over 32868 591 -> 70,
// 17 over 3017 61 -> 20, 1000 over 10000 188 -> 140; 8 / 2 heads, causal 2048 rows 43 -> 28. Over 5090 calls of random
// sizes that it splits (chunks, causal, bidirectional and prefix-causal rows) the time is 0.40 of the unsplit call's on
// the average and more than 1.02 of it in 11 (1.11 at most). Not split: prefix-causal calls whose item across
// `block` keeps most of its keys in one piece (445 rows over 1125 keys from position 3, block 59: 33 us, split 45), causal 1531
// rows of 32 heads (192 items of 1 to 24 tiles, at most a piece a CU: by the estimate the chip's clock and the merge take
// back most of what the shorter path gives), causal 4096 rows (512 items, heavy and light in turn).
template <int D>
SplitPlan split_plan(const mako_attn_args* a, uint32_t cus)
{
    constexpr double kTileUs = D == 128 ? 1.25 : 0.8, kFullUs = D == 128 ? 0.5 : 0.2, kWgUs = 8, kTurnUs = 3;
    constexpr double kMergeUs = 5;
    constexpr uint32_t kMinTiles = 6;  // a piece
    constexpr size_t kMaxBytes = 128u << 20;
    SplitPlan best;
    const uint32_t group = a->heads / a->kv_heads;
    const uint32_t hq = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const uint32_t rows_wg = 256 / hq, n_hg = a->heads / hq, n_qblk = (a->n_q + rows_wg - 1) / rows_wg;
    const uint64_t n_items = (uint64_t)n_hg * n_qblk;
    if (!cus || !a->n_k || !a->n_q || n_items > 4ull * cus || n_qblk > kSplitBlocks ||
        (uint64_t)a->q_pos0 + a->n_q + 256 > 0xffffffffull)
        return best;
    const auto tiles = [&](uint32_t qb) { return item_tiles(a, rows_wg, qb); };
    const uint32_t nt = tiles(n_qblk - 1);
    if (nt < 2 * kMinTiles)
        return best;
    const bool even = 2 * tiles(0) > nt;
    uint64_t total = 0;
    for (uint32_t qb = 0; qb < n_qblk; ++qb)
        total += (uint64_t)n_hg * tiles(qb);
    // the busiest CU's tiles: whole rounds of equal items with the longest among them, or a CU's share or the longest
    const auto path = [&](uint64_t n, double equal, double longest) {
        return even ? (double)((n - 1) / cus) * equal + longest : std::max(longest, (double)total / cus);
    };
    const double full_us = kFullUs * total / cus;
    double best_us = 0.85 * (kTileUs * path(n_items, nt, nt) + full_us + kWgUs);
    if (kTileUs * total / cus + full_us + kWgUs + kMergeUs >= best_us)
        return best;  // an even share and a merge are no shorter
    for (uint32_t np = 2; np <= 16 && nt / np >= kMinTiles; ++np) {
        SplitPlan s;
        s.piece_tiles = (nt + np - 1) / np;
        s.pieces = np;
        s.o_bytes = ((size_t)np * a->n_q * a->heads * D * 4 + 255) / 256 * 256;
        s.bytes = s.o_bytes + (size_t)np * a->heads * a->n_q * 4;
        if (s.bytes > kMaxBytes)
            break;
        uint64_t n = 0, merged = 0;  // pieces; pieces' rows the merge reads
        uint32_t longest = 0;        // tiles: an item with rows on both sides of `block` has a long last piece (Pieces)
        s.row0 = a->n_q;
        for (uint32_t qb = 0; qb < n_qblk; ++qb) {
            const Pieces pc(tiles(qb), first_keys(a, qb * rows_wg), s.piece_tiles);
            n += (uint64_t)n_hg * pc.np;
            longest = std::max(longest, pc.nt - pc.start(pc.np - 1));
            if (pc.np > 1) {
                merged += (uint64_t)pc.np * rows_wg * a->heads;
                s.row0 = std::min(s.row0, qb * rows_wg);
            }
        }
        // (the lists deal equal pieces evenly; of unequal ones a second round would put two long ones on a CU)
        if (!even && n > cus)
            continue;
        const double us = kTileUs * path(n, s.piece_tiles, std::max(longest, s.piece_tiles)) + full_us + kWgUs + kTurnUs * (double)((n - 1) / cus) +
                          kMergeUs + merged * D * 4.0 / 4.5e6;
        if (us < best_us) {
            best_us = us;
            best = s;
        }
    }
    return best;
}

}  // namespace

// The bytes flash_fwd_r64's split grid keeps its pieces in for this call (0: it runs unsplit). Only an offer: with
// less, or none, the call runs unsplit.
template <int D>
size_t fwd64_workspace(const mako_attn_args* a)
{
    const SplitPlan s = split_plan<D>(a, device_cus());
    return s.pieces > 1 ? s.bytes : 0;
}
template size_t fwd64_workspace<128>(const mako_attn_args*);
template size_t fwd64_workspace<64>(const mako_attn_args*);

// Launches flash_fwd_r64 for heads of D (128 or 64) on stream s: one launch with no workspace (K and V are staged from
// their rows), or the split grid and its merge where split_plan finds it faster and work has the memory (a stream that
// captures, or a caller without a workspace, keeps the one launch). Returns 1 when launched, 0 (launching nothing) when
// a size does not fit the kernel's 32-bit buffer offsets (the caller then uses flash_fwd).
template <class T, class TO, int D>
int launch_fwd64(const mako_attn_args* a, float scale_log2, const void* q, const void* k, const void* v, void* o,
                 float* lse, hipStream_t s, const Workspace& work)
{
    const uint32_t group = a->heads / a->kv_heads;
    const uint32_t hq = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const uint32_t rows_wg = 256 / hq;
    const uint32_t n_qblk = (a->n_q + rows_wg - 1) / rows_wg;
    if (!fwd64_fits<D>(a, sizeof(TO)))
        return 0;
    const uint32_t n_vt = (a->n_k + 63) / 64, n_hg = a->heads / hq, n_items = n_hg * n_qblk;
    const uint32_t cus = device_cus();
    const SplitPlan sp = split_plan<D>(a, cus);
    char* const ws = sp.pieces > 1 ? static_cast<char*>(work.try_get(kWsPieces, sp.bytes, s)) : nullptr;
    const Fwd64Params p{q, k, v, o, lse, a->n_q, a->q_pad, a->n_k, a->k_pad, a->heads, a->kv_heads, a->q_pos0,
                        a->block, a->width, scale_log2, group, hq, rows_wg, n_qblk, n_hg, n_vt, n_items};
    if (ws) {
        SplitParams ps;
        static_cast<Fwd64Params&>(ps) = p;
        ps.piece_tiles = sp.piece_tiles;
        ps.po = reinterpret_cast<float*>(ws);
        ps.pl = reinterpret_cast<float*>(ws + sp.o_bytes);
        uint32_t n = 0;
        for (uint32_t i = 0; i < kSplitBlocks; ++i) {
            if (i < n_qblk)
                n += (item_tiles(a, rows_wg, n_qblk - 1 - i) + sp.piece_tiles - 1) / sp.piece_tiles;
            ps.ends[i] = i < n_qblk ? (uint16_t)n : 0xffff;
        }
        hipLaunchKernelGGL((flash_fwd_r64<T, TO, D, true>), dim3(std::min(n * n_hg, cus)), dim3(256), 0, s, ps);
        const uint64_t rows = (uint64_t)(a->n_q - sp.row0) * a->heads, per = 1024 / D;
        hipLaunchKernelGGL((merge_pieces<TO, D>), dim3((uint32_t)((rows + per - 1) / per)), dim3(256), 0, s, ps,
                           sp.row0);
        return 1;
    }
    const uint32_t grid = std::min<uint32_t>(n_items, std::max<uint32_t>(1, cus));
    hipLaunchKernelGGL((flash_fwd_r64<T, TO, D, false>), dim3(grid), dim3(256), 0, s, p);
    return 1;
}

#define MAKO_FWD64_INSTANCE(T, TO, D)                                                                            \
    template int launch_fwd64<T, TO, D>(const mako_attn_args*, float, const void*, const void*, const void*, void*, \
                                        float*, hipStream_t, const Workspace&);
MAKO_FWD64_INSTANCE(__bf16, float, 128)
MAKO_FWD64_INSTANCE(__bf16, __bf16, 128)
MAKO_FWD64_INSTANCE(_Float16, float, 128)
MAKO_FWD64_INSTANCE(_Float16, _Float16, 128)
MAKO_FWD64_INSTANCE(__bf16, float, 64)
MAKO_FWD64_INSTANCE(__bf16, __bf16, 64)
MAKO_FWD64_INSTANCE(_Float16, float, 64)
MAKO_FWD64_INSTANCE(_Float16, _Float16, 64)
#undef MAKO_FWD64_INSTANCE

// The V^T images flash_fwd_d256 stages from: kv_heads x ceil(n_k / 64) tiles of 32 KiB (0 when the kernel does not
// take the call).
size_t d256_workspace(const mako_attn_args* a)
{
    return d256_fits(a) ? (size_t)a->kv_heads * ((a->n_k + 63) / 64) * R64<256>::kVTile : 0;
}

// Launches vt_image<T, 256> and flash_fwd_d256 on stream s, the V^T images in the call's workspace (work), or already
// written at vt_ready. Returns 1 when launched, 0 (launching nothing) when a size does not fit the kernel's 32-bit
// buffer offsets (the caller then uses flash_fwd_wide), -1 when the workspace could not be had (the error recorded).
template <class T, class TO>
int launch_fwd_d256(const mako_attn_args* a, float scale_log2, const void* q, const void* k, const void* v, void* o,
                    float* lse, hipStream_t s, const void* vt_ready, const Workspace* work)
{
    using L = R64<256>;
    const uint32_t group = a->heads / a->kv_heads;
    const uint32_t hq = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
    const uint32_t rows_wg = 128 / hq;
    const uint32_t n_qblk = (a->n_q + rows_wg - 1) / rows_wg;
    const uint32_t n_vt = (a->n_k + 63) / 64;
    if (!d256_fits(a))
        return 0;
    const size_t need = (size_t)a->kv_heads * n_vt * L::kVTile;
    const void* vt = vt_ready;
    if (!vt_ready && need) {
        void* ws = work->get(need, s);
        if (!ws)
            return -1;
        vt = ws;
        hipLaunchKernelGGL((vt_image<T, 256>), dim3(n_vt, a->kv_heads), dim3(256), 0, s, static_cast<const T*>(v),
                           static_cast<uint32_t*>(ws), a->n_k, a->k_pad, n_vt);
    }
    const Fwd64Params p{q, k, vt, o, lse, a->n_q, a->q_pad, a->n_k, a->k_pad, a->heads, a->kv_heads, a->q_pos0,
                        a->block, a->width, scale_log2, group, hq, rows_wg, n_qblk, a->heads / hq, n_vt,
                        a->heads / hq * n_qblk};
    hipLaunchKernelGGL((flash_fwd_d256<T, TO>), dim3(a->heads / hq, n_qblk), dim3(256), 0, s, p);
    return 1;
}

#define MAKO_D256_INSTANCE(T, TO)                                                                                \
    template int launch_fwd_d256<T, TO>(const mako_attn_args*, float, const void*, const void*, const void*, void*, \
                                        float*, hipStream_t, const void*, const Workspace*);
MAKO_D256_INSTANCE(__bf16, float)
MAKO_D256_INSTANCE(__bf16, __bf16)
MAKO_D256_INSTANCE(_Float16, float)
MAKO_D256_INSTANCE(_Float16, _Float16)
#undef MAKO_D256_INSTANCE

}  // namespace mako
