// Tiled attention forward on the bf16/fp16 MFMA for gfx950: variable-length (token-major) prefill
// over dense or paged K/V, and kvcache calls whose query block is too tall for the decode kernel.
//
// Stands in for the reference's FAInfer kernel in TND layout (csrc/ascend910/flash_attn_npu/
// mha_fwd_kvcache.cpp:436-970 with per-sequence offsets :469-475,505-507; host mha_varlen_fwd,
// flash_api.cpp:848-1089).  Where the reference ping-pongs S, P and O_tmp between its matrix and
// vector cores through global memory, everything between the K/V tile loads and the final store
// stays in registers here:
//   * one workgroup = 128 query rows of one (sequence, q head); 4 waves x 32 rows.  Under GQA short
//     query blocks, and causal launches of many tiles, are packed instead (p.pack = group): the 128 rows are
//     (query, head of the group) pairs of one kv head, query-major, so a 16-token block of an 8-head group
//     fills a tile and K/V are read once per kv head (the reference packs heads the same way,
//     flash_api.cpp:33-95), and a causal tile's keys end closer behind its queries (prefill_tiling());
//   * K/V tiles of 64 keys are fetched once per workgroup, 16 bytes per lane, straight from global memory
//     into LDS (no register holds them and no LDS store instruction moves them: such a store keeps the
//     wave from issuing anything else for ~50 cycles, and the tile stores were a tenth of the kernel's
//     time), swizzled so that the operand reads are conflict free (the lane that fills a piece's place in
//     LDS fetches the piece that belongs there); K tiles double-buffered, V tiles as far as LDS allows;
//   * S^T = K Q^T and O^T = V^T P^T on the 32x32x16 MFMA: a query row is one lane column in both
//     products, so the running max / sum / rescale never leave the lane (one xor-32 exchange);
//   * V^T operands come straight from the transposing LDS read (ds_read_b64_tr_b16);
//   * key tiles outside the causal / window range of the 128-row block are never loaded.
#include <type_traits>

#include "fa_device.h"
#include "fa_kernels.h"

namespace fa {

constexpr int kBM = 128;  // query rows per workgroup
constexpr int kBN = 64;   // keys per tile

template <int D> struct PrefillCfg {
    static constexpr int kKSteps = D / 16;        // MFMA k-steps of QK^T
    static constexpr int kMT = D / 32;            // 32-column tiles of O^T
    static constexpr int kChunks = D / 8;         // 16-byte pieces per row
    static constexpr int kRowBytes = D * 2;
    static constexpr int kTileBytes = kBN * kRowBytes;
    static constexpr int kVBufs = D == 128 ? 1 : 2;                // (see prefill_wgs_resident)
    // A tile is filled by loads that go from global memory straight to LDS (global_load_lds_dwordx4): one instruction
    // of a wave fills 64 consecutive 16-byte pieces, lane l the piece at the instruction's LDS base + 16 l, from
    // whatever address the lane names.  The four waves share the pieces of a tile, instruction by instruction.
    static constexpr int kLoads = kBN * kChunks / 256;             // per wave and tile (K or V)
    static constexpr int kLoadRows = 256 / kChunks;                // rows between a wave's consecutive loads
    static_assert(kBN * kChunks % 256 == 0, "whole instructions per wave");
    // Swizzles that spread the operand reads over all banks (256 bytes wide).  K: 16 rows of an operand are read 16
    // bytes each, so their pieces have to stand in 16 different places; V: the transposing read takes 64 bytes (32
    // columns) of each of 4 rows.  Rows of 128 bytes lie two in a line of banks and change place every other row.
    static __device__ __forceinline__ int k_place(int row, int piece) { return piece ^ (D == 64 ? (row >> 1) & 7 : row & 15); }
    static __device__ __forceinline__ int v_place(int row, int piece) { return piece ^ ((D == 64 ? (row >> 1) & 1 : row & 3) << 2); }
    static constexpr int kPatterns = D == 256 ? 2 : 1;             // loads after which the places of a lane's pieces repeat
};

// K tiles: the one being read and the one on its way; V tiles likewise, or a single one (kVBufs).  Starts at a multiple of two
// tiles: the buffer, and the place in a row, are chosen by XOR.
template <int D> struct PrefillTileLds {
    uint8_t k[2][PrefillCfg<D>::kTileBytes];
    uint8_t v[PrefillCfg<D>::kVBufs][PrefillCfg<D>::kTileBytes];
};

// EXT: packed heads and / or a split of the keys (p.pack, p.nsplits); without it both are compiled out
// One 128-row block of one (sequence, key range, kv head, q head) of the launch: `bid` is its place in the
// launch's order.  n_long < 0: the units are the launch's batch rows; otherwise they are the first n_long entries of
// p.long_ids (the sequences the tiled kernel computes, listed on the device).
// PART: the head dimension p.headdim is below D: pieces of the q / k / v rows behind it are zeros that nobody loads,
// k-steps and output tiles that only see such pieces are skipped, and the stores stop at the head dimension.
template <typename T, int D, bool PAGED, bool SOFTCAP, bool EXT, bool PART>
__device__ __forceinline__ void prefill_block(const PrefillParams &p, const unsigned bid, const int n_long, PrefillTileLds<D> &lds) {
    using Cfg = PrefillCfg<D>;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // (a kernel that walks several blocks would keep what is made of it through all of them)
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lh = lane >> 5;   // half: MFMA k-slot
    const int ln = lane & 31;   // MFMA row / column
    const int hd = PART ? p.headdim : D;

    const int nsplits = EXT ? max(p.nsplits, 1) : 1;
    const int heads_per_unit = (EXT && p.pack > 1) ? 1 : p.group;
    const bool listed = EXT && n_long >= 0;
    const int n_units = (listed ? n_long : p.batch) * nsplits * p.nheads_k;
    const int units8 = listed ? (n_units + 7) / 8 * 8 : p.units8;
    const PrefillPlace place = prefill_place(bid, p.num_mb, EXT ? p.mb_run : 1, units8, heads_per_unit);
    const int mb = place.mb, unit = place.unit, head_in_unit = place.head;
    if (unit >= n_units) return;
    const int z = unit / p.nheads_k;
    const int hk = unit - z * p.nheads_k;
    const int zb = z / nsplits;
    const int split = z - zb * nsplits;
    // Lengths and tables do not change while the kernel runs and are read at the same place by every lane: scalar loads, which leave
    // what follows from them in scalar registers.  They are asked for together, a trip to memory for all of them.
    auto constant = [](const int32_t *ptr, int i) -> int { return ((const __attribute__((address_space(4))) int32_t *)(uintptr_t)ptr)[i]; };
    auto scalar = [](int x) -> int { return __builtin_amdgcn_readfirstlane(x); };   // (values out of LDS)
    const int b = listed ? constant(p.long_ids, zb) : zb;
    int q0, Sq, k0 = 0, Sk;
    if constexpr (PAGED) {
        Sk = constant(p.seqused_k, b);
    } else {
        k0 = constant(p.cu_seqlens_k, b);
        Sk = constant(p.cu_seqlens_k, b + 1);
    }
    if (p.cu_seqlens_q) {
        q0 = constant(p.cu_seqlens_q, b);
        Sq = constant(p.cu_seqlens_q, b + 1) - q0;
    } else {
        q0 = 0;
        Sq = p.seqlen_q_fixed;
    }
    if (EXT && Sq >= 1 && Sq <= p.skip_short) return;   // the decode kernels compute this sequence
    // tile row R is query R / pg of head h_base + R % pg.  pg is the launch's (every block packs the heads
    // of its group, or none does) unless the launch lets short blocks pack on their own: a block whose
    // (query, head) rows take at most three quarters of the tiles its heads would take one by one is
    // computed by the tiles of its first head alone, the tiles of the other heads leave
    int pg = EXT ? p.pack : 1;
    if (EXT && p.pack_short && pg == 1 && p.group > 1) {
        const int packed = (Sq * p.group + kBM - 1) / kBM;
        const int plain = p.group * ((Sq + kBM - 1) / kBM);
        if (packed * 4 <= plain * 3 && packed <= p.num_mb) {
            if (head_in_unit != 0) return;
            pg = p.group;
        }
    }
    const int h_base = hk * p.group + ((pg > 1) ? 0 : head_in_unit);
    if constexpr (PAGED) {
        Sk = min(Sk + p.seqlen_k_add, p.max_blocks * p.page_size);
    } else {
        Sk -= k0;
        if (p.seqused_k) Sk = max(0, min(Sk, constant(p.seqused_k, b)));   // only the first seqused_k[b] keys of the sequence are used
    }
    // window normalisation: the varlen host passes max_seqlen_k as the reference does
    // (flash_api.cpp:938-943); the kvcache layout has the lengths on the device only, so the batch
    // maximum is reduced here when a window was requested
    int wl = p.window_left, wr_eff = p.window_right;
    int norm_m = p.window_norm_m;
    if constexpr (PAGED) {
        if (norm_m <= 0 && (wl >= 0 || wr_eff >= 0)) norm_m = scalar(block_max_keys(p.seqused_k, p.batch, p.seqlen_k_add));
    }
    if (norm_m <= 0) norm_m = max(Sk, 1);
    normalize_window(wl, wr_eff, p.causal, norm_m);
    int batch_max = 0;
    if constexpr (PAGED) {
        if (nsplits > 1) batch_max = scalar(min(block_max_keys(p.seqused_k, p.batch, p.seqlen_k_add), p.max_blocks * p.page_size));
    }
    const int n_rows = Sq * pg;
    const int R0 = mb * kBM;
    if (R0 >= n_rows) return;
    const int off = Sk - Sq;

    // split of the unit's visible keys: the same cut as the decode kernels' grid mode, so that the
    // same combine kernel merges the partials
    int range_lo = 0, range_hi = Sk;
    bool whole = true;
    int64_t slot = 0;
    if (nsplits > 1) {
        const int sk = adaptive_split_keys(batch_max, nsplits);
        const KeyRanges kr = key_ranges(Sq, Sk, wl, wr_eff, sk, nsplits);
        if (split >= kr.count) return;
        if (kr.hi > kr.lo) {
            range_lo = kr.begin(split, sk);
            range_hi = kr.end(split, sk);
        }
        whole = kr.count == 1;
        slot = ((int64_t)b * p.nheads_k + hk) * nsplits + split;
    }

    // Tile row R0 + i is query `pos` of head `head`; rows past the end (ok: false) repeat the last one and are dropped.  Worked out
    // where it is needed: kept through the loop, it would take registers that the operands need.
    const int r_lo = R0 / pg;                                // query positions of the block: r_lo .. r_hi
    const int r_hi = (min(n_rows, R0 + kBM) - 1) / pg;
    const uint32_t pg_inv = (EXT && pg > 1) ? 0xffffffffu / (uint32_t)pg + 1u : 0u;   // x / pg = the upper half of x * pg_inv for x < pg + 128
    struct TileRow {
        int pos, head;
        bool ok;
    };
    auto tile_row = [&](int i) -> TileRow {
        const int R = min(R0 + i, n_rows - 1);
        TileRow t;
        t.ok = R0 + i < n_rows;
        t.pos = (EXT && pg > 1) ? r_lo + (int)__umulhi((uint32_t)(R - r_lo * pg), pg_inv) : R;
        t.head = h_base + (R - t.pos * pg);
        return t;
    };
    auto this_lane = [&]() -> int {                          // (found out anew, so that it need not be kept either)
        int l;
        asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
        return l;
    };
    auto my_row = [&](int l) -> TileRow { return tile_row(wave * 32 + (l & 31)); };   // the row of lane l's column
    auto lse_of = [&](const TileRow &t) -> float * { return p.lse + (int64_t)b * p.lse_stride_b + (int64_t)t.head * p.lse_stride_h + q0 + t.pos; };

    // key range the whole block (query positions r_lo .. r_hi) can see
    int k_lo = 0, k_hi = Sk;
    if (wl >= 0) k_lo = max(0, r_lo + off - wl);
    if (wr_eff >= 0) k_hi = min(Sk, r_hi + off + wr_eff + 1);
    k_lo = max(k_lo, range_lo);
    k_hi = max(min(k_hi, range_hi), 0);
    // where a row goes when the unit is cut: row (query, head of the group) of the slot
    auto part_of = [&](const TileRow &t) -> int64_t {
        // kvcache layout: (batch row, kv head, range, query x head of the group); token-major q: (token, head, range)
        return p.cu_seqlens_q ? ((int64_t)(q0 + t.pos) * p.nheads + t.head) * nsplits + split
                              : slot * p.rows + (int64_t)t.pos * p.group + (t.head - hk * p.group);
    };

    if (k_hi <= k_lo) {
        // nothing visible for the whole block: out = 0, lse = +inf
        const TileRow t = my_row(lane);
        if (t.ok && whole) {
            uint16_t *o_row = reinterpret_cast<uint16_t *>(p.out) + (int64_t)b * p.o_stride_b + (int64_t)t.head * p.o_stride_h +
                              (int64_t)(q0 + t.pos) * p.o_stride_t;
            for (int c = lh * (D / 2); c < min((lh + 1) * (D / 2), hd); c += 8) store16(o_row + c, u32x4_t{0, 0, 0, 0});
            if (lh == 0) *lse_of(t) = INFINITY;
        } else if (t.ok) {
            float *part_row = p.o_partial + part_of(t) * D;
            for (int c = lh * (D / 2); c < (lh + 1) * (D / 2); c += 4) *reinterpret_cast<float4 *>(part_row + c) = make_float4(0.f, 0.f, 0.f, 0.f);
            if (lh == 0) p.lse_partial[part_of(t)] = -INFINITY;
        }
        return;
    }

    // bounds that decide, per wave, whether a tile needs element masks
    const int rw0 = min(R0 + wave * 32, n_rows - 1) / pg;        // first and last query position of the wave
    const int rw1 = (min(n_rows, R0 + wave * 32 + 32) - 1) / pg;
    const int wave_klo_max = max(range_lo, (wl >= 0) ? max(0, rw1 + off - wl) : 0);
    // the keys that any row of the wave sees: halves of a tile beyond them are left out
    const int wave_klo_first = max(range_lo, (wl >= 0) ? max(0, rw0 + off - wl) : 0);
    const int wave_khi_last = min(range_hi - 1, (wr_eff >= 0) ? min(Sk - 1, rw1 + off + wr_eff) : Sk - 1);
    const int wave_khi_min = min(range_hi - 1, (wr_eff >= 0) ? min(Sk - 1, rw0 + off + wr_eff) : Sk - 1);

    // Q^T operand: lane (lh, ln) holds row ln, elements t*16 + lh*8 .. +7
    u32x4_t qreg[Cfg::kKSteps];
    {
        const TileRow row = my_row(lane);
        const uint16_t *src = reinterpret_cast<const uint16_t *>(p.q) + (int64_t)b * p.q_stride_b + (int64_t)row.head * p.q_stride_h +
                              (int64_t)(q0 + row.pos) * p.q_stride_t + lh * 8;
#pragma unroll
        for (int t = 0; t < Cfg::kKSteps; ++t) {
            if (PART && t * 16 + lh * 8 >= hd) {
                qreg[t] = u32x4_t{0, 0, 0, 0};
                continue;
            }
            qreg[t] = load16(src + t * 16);
            if (!row.ok) qreg[t] = u32x4_t{0, 0, 0, 0};
        }
    }

    // ---- K/V tile fetch ---------------------------------------------------------------------
    const uint16_t *kbase = reinterpret_cast<const uint16_t *>(p.k) + (int64_t)hk * p.k_stride_h;
    const uint16_t *vbase = reinterpret_cast<const uint16_t *>(p.v) + (int64_t)hk * p.v_stride_h;
    const int32_t *bt_row = PAGED ? p.block_table + (int64_t)b * p.bt_stride_b : nullptr;

    // Load i of this wave covers the LDS pieces 64 (wave + 4i) .. + 63 of the tile, piece = (row, place in the row); a row's
    // place c' holds the row's piece k_place(row, c') or v_place(row, c') (their own inverses).
    // Rows past the last key re-read the last key (never memory nobody wrote; they are masked); with PART the pieces
    // behind the head dimension are not loaded: their places hold the zeros written when the block started.
    auto t_row = [&](int l) -> int { return (64 * wave + l) / Cfg::kChunks; };   // lane l's row of load 0; load i: kLoadRows * i rows on
    uint32_t k_off[Cfg::kPatterns], v_off[Cfg::kPatterns];    // offsets of load 0 (1) in an interior tile: one wave-uniform base serves all lanes
    bool k_on[Cfg::kPatterns], v_on[Cfg::kPatterns];
    auto col_of = [&](bool is_k, int i, int l) -> int {       // its piece in the row of load i
        const int c = l % Cfg::kChunks, row = t_row(l) + i * Cfg::kLoadRows;
        return is_k ? Cfg::k_place(row, c) : Cfg::v_place(row, c);
    };
#pragma unroll
    for (int i = 0; i < Cfg::kPatterns; ++i) {
        k_on[i] = !PART || col_of(true, i, lane) * 8 < hd;
        v_on[i] = !PART || col_of(false, i, lane) * 8 < hd;
        k_off[i] = (uint32_t)t_row(lane) * (uint32_t)p.k_stride_t * 2u + col_of(true, i, lane) * 16;
        v_off[i] = (uint32_t)t_row(lane) * (uint32_t)p.v_stride_t * 2u + col_of(false, i, lane) * 16;
    }
    auto lds_of = [](const void *ptr) -> uint32_t { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void *)ptr; };
    // The loads are written out: the compiler would wait for such a load in front of every LDS read that follows (it
    // cannot tell the two buffers apart).  tiles_landed() is the wait that orders them.
    auto load_lds_base = [&](uint32_t lds, uint32_t off, const uint8_t *base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
    };
    auto load_lds_addr = [&](uint32_t lds, const void *addr) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(addr) : "memory", "m0");
    };
    auto uniform = [](const uint8_t *ptr) -> const uint8_t * {   // (for the compiler; it is)
        const uint64_t x = reinterpret_cast<uint64_t>(ptr);
        return reinterpret_cast<const uint8_t *>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32 |
                                                 (uint32_t)__builtin_amdgcn_readfirstlane((int)x));
    };
    auto tiles_landed = [&]() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    // Where the tiles of a paged cache are.  A page holds a multiple of 32 keys (or, a page per sequence, all of them), so each half of
    // a tile lies in one page, and the cursor keeps the addresses of both halves.  Inside a page a step moves them on by 64 rows;
    // where a page ends they are made from the table, whose next two entries were asked for when the page before began: by scalar
    // loads, which nobody has to wait for behind the tiles on their way.  All of it is scalar work of every wave: the addresses made
    // anew for every tile cost a paged launch 8 % (4 x 2048 tokens over 8 K keys 1136 us against 1048 dense, now 1015 against 985);
    // a page looked up per row, with 32-row pages, a third (8 x 51 tokens over 4481..8962 keys, d = 64, 106 us against 79 now).
    const int page_rows = !PAGED || p.max_blocks == 1 ? INT32_MAX : p.page_size;
    auto table = [&](int page) -> int { return constant(bt_row, min(page, p.max_blocks - 1)); };
    struct Cursor {
        const uint8_t *k[2], *v[2];     // first row of each half
        int row[2], page;               // place of the halves in their pages (kept for the second one), its page
        int id, ahead[2];               // table entry of that page and of the next two
    };
    const int64_t k_row = p.k_stride_t * 2, v_row = p.v_stride_t * 2;   // bytes
    auto set_half = [&](Cursor &c, int h, int id) {
        const int64_t block = min(max(__builtin_amdgcn_readfirstlane(id), 0), p.num_blocks - 1);
        c.k[h] = uniform(reinterpret_cast<const uint8_t *>(kbase) + c.row[h] * k_row + block * p.k_stride_block * 2);
        c.v[h] = uniform(reinterpret_cast<const uint8_t *>(vbase) + c.row[h] * v_row + block * p.v_stride_block * 2);
    };
    auto first_tile = [&](int kt) -> Cursor {
        Cursor c = {};
        if constexpr (PAGED) {
            const int page0 = kt * kBN / page_rows;
            c.page = (kt * kBN + 32) / page_rows;
            c.row[0] = kt * kBN - page0 * page_rows;
            c.row[1] = kt * kBN + 32 - c.page * page_rows;
            c.id = table(c.page);
            c.ahead[0] = table(c.page + 1);
            c.ahead[1] = table(c.page + 2);
            set_half(c, 0, table(page0));
            set_half(c, 1, c.id);
        }
        return c;
    };
    auto advance = [&](Cursor &c) {
        if constexpr (!PAGED) return;
        if (c.row[1] + kBN < page_rows) {
            // (the first half may have come from the page before)
            c.row[1] += kBN;
            c.k[1] += kBN * k_row;
            c.v[1] += kBN * v_row;
            c.k[0] = c.k[1] - 32 * k_row;
            c.v[0] = c.v[1] - 32 * v_row;
            return;
        }
        // the halves stand 32 and 64 rows behind the second half of the tile before
        const int old = c.page;
        int at = c.row[1];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            at += 32;
            if (at >= page_rows) {
                at -= page_rows;
                ++c.page;
            }
            c.row[h] = at;
            set_half(c, h, c.page == old ? c.id : c.ahead[c.page == old + 1 ? 0 : 1]);
        }
        if (c.page != old) {
            c.id = c.ahead[c.page == old + 1 ? 0 : 1];
            c.ahead[0] = table(c.page + 1);
            c.ahead[1] = table(c.page + 2);
        }
    };
    // K (IS_K) or V tile kt into its buffer
    auto fetch = [&](auto is_k_c, int kt, const uint8_t *const (&half)[2]) {
        constexpr bool IS_K = decltype(is_k_c)::value;
        const uint32_t dst = lds_of(IS_K ? &lds.k[kt & 1][0] : &lds.v[kt & (Cfg::kVBufs - 1)][0]) + (uint32_t)wave * 1024u;
        const int64_t row_bytes = IS_K ? k_row : v_row;
        const uint32_t(&off)[Cfg::kPatterns] = IS_K ? k_off : v_off;
        const bool(&on)[Cfg::kPatterns] = IS_K ? k_on : v_on;
        const int last = Sk - 1 - kt * kBN;                   // last written key relative to the tile (>= 0)
        static_assert(32 % Cfg::kLoadRows == 0, "a load lies in one half");
        const uint8_t *dense = nullptr;                       // (two multiplications: running pointers would take scalar registers)
        if constexpr (!PAGED) dense = reinterpret_cast<const uint8_t *>(IS_K ? kbase : vbase) + (k0 + kt * kBN) * row_bytes;
        auto from = [&](int h) -> const uint8_t * { return PAGED ? half[h] : dense + 32 * h * row_bytes; };
        if (last >= kBN - 1) {
#pragma unroll
            for (int i = 0; i < Cfg::kLoads; ++i) {
                const int row = i * Cfg::kLoadRows, h = row / 32;   // first row of the load over all waves
                if (on[i % Cfg::kPatterns]) load_lds_base(dst + i * 4096u, off[i % Cfg::kPatterns], from(h) + (row - 32 * h) * row_bytes);
            }
        } else {
            // the ragged end of a sequence: rows past the last key re-read it
            const int l = this_lane();
#pragma unroll
            for (int i = 0; i < Cfg::kLoads; ++i) {
                const int row = i * Cfg::kLoadRows, h = last < 32 * (row / 32) ? 0 : row / 32;
                if (on[i % Cfg::kPatterns])
                    load_lds_addr(dst + i * 4096u, from(h) + (min(t_row(l) + row, last) - 32 * h) * row_bytes + col_of(IS_K, i, l) * 16);
            }
        }
    };
    if constexpr (PART) {
        // the places of the pieces that nobody loads
        for (int i = tid * 16; i < (2 + Cfg::kVBufs) * Cfg::kTileBytes; i += 256 * 16) *reinterpret_cast<u32x4_t *>(&lds.k[0][0] + i) = u32x4_t{0, 0, 0, 0};
        __syncthreads();
    }

    float m_run = -INFINITY, l_run = 0.f;
    float16_t o_acc[Cfg::kMT];
#pragma unroll
    for (int t = 0; t < Cfg::kMT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o_acc[t][r] = 0.f;

    // (uniform, which the compiler cannot see behind the batch maximum that comes out of LDS)
    const int kt_begin = __builtin_amdgcn_readfirstlane(k_lo / kBN);
    const int kt_end = __builtin_amdgcn_readfirstlane((k_hi + kBN - 1) / kBN);
    const bool wave_live = __builtin_amdgcn_readfirstlane(R0 + wave * 32 < n_rows);
    const std::true_type K_TILE{};
    const std::false_type V_TILE{};
    // Step kt: behind the barrier in front of it K tile kt is there and every wave has used K tile kt - 1 and V tile kt - 1.  With
    // one V buffer the V tile of the step itself is asked for here, and waited for (with a barrier) behind the softmax; with two
    // it was asked for a step ago.
    auto landed_but = [&](auto n_c) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n_c)::value) : "memory"); };
    auto barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    Cursor next = first_tile(kt_begin);
    fetch(K_TILE, kt_begin, next.k);
    if (Cfg::kVBufs == 2) fetch(V_TILE, kt_begin, next.v);
    const uint8_t *v_here[2] = {next.v[0], next.v[1]};       // V tile kt
    advance(next);
    tiles_landed();
    barrier();

    float16_t s[2];                 // scores of a tile: keys 0-31 and 32-63
    u32x4_t ka[Cfg::kKSteps][2];
    // LDS addresses of this lane's operand pieces in the tile's buffer: K row ln, piece lh (k-step t: XOR t << 5), V row tr_row, its 8
    // bytes of column tile 0 (tile t: XOR t << 6)
    const int tr_row = 4 * lh + ((lane & 15) >> 2);
    uint32_t k_at = lds_of(&lds.k[0][0]) + (uint32_t)ln * Cfg::kRowBytes + ((uint32_t)Cfg::k_place(ln, lh) << 4);
    uint32_t v_at = lds_of(&lds.v[0][0]) + (uint32_t)tr_row * Cfg::kRowBytes +
                            ((uint32_t)Cfg::v_place(tr_row, ((lane >> 4) & 1) * 2 + ((lane >> 1) & 1)) << 4) + (uint32_t)(lane & 1) * 8u;
    k_at += (uint32_t)(kt_begin & 1) * Cfg::kTileBytes;
    v_at += (uint32_t)(kt_begin & (Cfg::kVBufs - 1)) * Cfg::kTileBytes;
    auto read_k = [&](int t, int halves) {
#pragma unroll
        for (int tt = 0; tt < halves; ++tt)
            ka[t][tt] = *(const __attribute__((address_space(3))) u32x4_t *)(uintptr_t)((k_at ^ (uint32_t)(t << 5)) + tt * 32 * Cfg::kRowBytes);
    };
    constexpr int kPf = 2;          // operand reads run kPf k-steps ahead of the MFMAs that use them
    const float16_t zero16 = {};
    // Packed tiles and key ranges end anywhere in a key tile, and a wave's 128 / 4 / group queries end before those of the block:
    // a half of a tile that no row of the wave sees is left out (its weights are zero).  80 x 3..350 tokens, 28q/4kv 77.8 -> 73.8 us,
    // 16 x 512..4096, 32q/8kv 714 -> 705; without packing (one tile in 33 at 2050 keys) what it saves the second form of the step takes.
    constexpr bool kHalves = EXT;
    for (int kt = kt_begin; kt < kt_end; ++kt) {
        const bool more = kt + 1 < kt_end;
        if (Cfg::kVBufs == 1) fetch(V_TILE, kt, v_here);
        if (more) {
            fetch(K_TILE, kt + 1, next.k);
            if (Cfg::kVBufs == 2) fetch(V_TILE, kt + 1, next.v);
        }
        __builtin_amdgcn_sched_barrier(0);
        u32x4_t pk[2][2];
        const int tile0 = kt * kBN;
        // Halves of the tile (32 keys each, the first one or both) that some row of the wave sees.  A wave without any (its 32 rows
        // all lie past the block's end, as with a decode row among prompt chunks, or end in front of the tile) only helps to move
        // the tiles, and leaves the matrix pipe to the others.
        const int live = __builtin_amdgcn_readfirstlane(!wave_live || tile0 > wave_khi_last || tile0 + kBN <= wave_klo_first ? 0
                                                        : kHalves && tile0 + 32 > wave_khi_last                            ? 1
                                                                                                                           : 2);
        auto weights = [&](auto halves_c) {
            constexpr int H = decltype(halves_c)::value;
            // ---- S^T = K Q^T for the 32-key halves of the tile.  The wave in a matrix phase goes first: its MFMAs then issue
            // back to back and the vector work of the SIMD's other waves fills the gaps between them
            __builtin_amdgcn_s_setprio(1);
            asm volatile("" : "+v"(k_at));   // (opaque: kept from step to step, the address of every operand would take a register)
#pragma unroll
            for (int t = 0; t < kPf; ++t) read_k(t, H);
#pragma unroll
            for (int t = 0; t < Cfg::kKSteps; ++t) {
                if (PART && t * 16 >= hd) break;   // wave-uniform; at least D/2 columns are live
                if (t + kPf < Cfg::kKSteps) read_k(t + kPf, H);
#pragma unroll
                for (int tt = 0; tt < H; ++tt) s[tt] = mfma32<T>(ka[t][tt], qreg[t], t == 0 ? zero16 : s[tt]);
                __builtin_amdgcn_sched_barrier(0);
            }

            __builtin_amdgcn_s_setprio(0);
            // ---- online softmax; lane column = query row, register r of half tt = key
            //      kt*64 + tt*32 + 8*(r/4) + 4*lh + r%4
            // wave-uniform by construction; made scalar so the two softmax paths stay separate branches
            const bool need_mask = __builtin_amdgcn_readfirstlane((tile0 < wave_klo_max) || (tile0 + kBN - 1 > wave_khi_min));
            // The scores are left unscaled where that can be (no softcap, positive scale): the maximum is taken on them as they
            // are, and the scale rides in the exponent's fused multiply-add.
            if constexpr (SOFTCAP) {
#pragma unroll
                for (int tt = 0; tt < H; ++tt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float y = s[tt][r] * p.softcap_pre;
                        const float e2 = __expf(2.f * y);
                        s[tt][r] = p.softcap_post * (1.f - 2.f / (e2 + 1.f));
                    }
            } else if (!(p.scale_log2 > 0.f)) {
#pragma unroll
                for (int tt = 0; tt < H; ++tt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[tt][r] *= p.scale_log2;
            }
            const float scale = (!SOFTCAP && p.scale_log2 > 0.f) ? p.scale_log2 : 1.f;
            if (need_mask) {
                // masked tile (the diagonal of a causal block, window edges, the ragged end): element r
                // of half tt is key tile0 + 4*lh + e(tt, r) with e a compile-time constant, so the
                // row's bounds are compared in tile coordinates; a side that cannot bite is skipped
                const int l = this_lane(), at = my_row(l).pos + off, first = tile0 + 4 * (l >> 5);
                const int lo_rel = max(range_lo, (wl >= 0) ? at - wl : 0) - first;
                const int hi_rel = min(range_hi - 1, (wr_eff >= 0) ? min(Sk - 1, at + wr_eff) : Sk - 1) - first;
#pragma unroll
                for (int tt = 0; tt < H; ++tt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int e = tt * 32 + 8 * (r >> 2) + (r & 3);
                        s[tt][r] = (e <= hi_rel) ? s[tt][r] : -INFINITY;
                    }
                if (__builtin_amdgcn_readfirstlane(tile0 < wave_klo_max)) {
#pragma unroll
                    for (int tt = 0; tt < H; ++tt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int e = tt * 32 + 8 * (r >> 2) + (r & 3);
                            s[tt][r] = (e >= lo_rel) ? s[tt][r] : -INFINITY;
                        }
                }
            }
            float mloc = -INFINITY;
#pragma unroll
            for (int tt = 0; tt < H; ++tt)
#pragma unroll
                for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, s[tt][r]);
            mloc *= scale;
            mloc = halves_max(mloc);
            // The accumulator rescale is skipped for the whole wave when no row of it saw a new maximum
            // (most tiles once a row is a few hundred keys in).  m_run is the running maximum times the scale, rounded, and
            // the exponent the fused s * scale - m_run: the largest P of a row is 1 but for that rounding (2^d, |d| at most
            // half a unit in the last place of m_run), in the weights, their sum and the LSE alike.
            const bool bump = mloc > m_run;   // false for fully hidden tiles
            if (__any(bump)) {
                const float m_new = bump ? mloc : m_run;
                const float m_new_use = (m_new == -INFINITY) ? 0.f : m_new;
                const float alpha = bump ? fast_exp2(m_run - m_new_use) : 1.f;
                m_run = m_new;
                l_run *= alpha;
#pragma unroll
                for (int t = 0; t < Cfg::kMT; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o_acc[t][r] *= alpha;
            }
            const float m_use = (m_run == -INFINITY) ? 0.f : m_run;
            float psum = 0.f;
#pragma unroll
            for (int tt = 0; tt < H; ++tt)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[tt][r] = fast_exp2(__builtin_fmaf(s[tt][r], scale, -m_use));
#pragma unroll
            for (int tt = 0; tt < H; ++tt) {
#pragma unroll
                for (int r = 0; r < 16; ++r) psum += s[tt][r];
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int u = 0; u < 4; ++u) pk[tt][ks][u] = pack2<T>(s[tt][8 * ks + 2 * u], s[tt][8 * ks + 2 * u + 1]);
            }
            l_run += psum;
        };
        if (live == 2) weights(std::integral_constant<int, 2>{});
        if (kHalves && live == 1) weights(std::integral_constant<int, 1>{});
        if (Cfg::kVBufs == 1) {
            // V tile kt (the loads of K tile kt + 1 behind it may still be on their way; with PART some of those are left out)
            if (more && !PART) landed_but(std::integral_constant<int, Cfg::kLoads>{}); else tiles_landed();
            barrier();
        }
        auto products = [&](auto halves_c) {
            constexpr int H = decltype(halves_c)::value;
            __builtin_amdgcn_s_setprio(1);
            // ---- O^T += V^T P^T, 16 keys per step.  The V^T operand comes from the transposing LDS read
            //      (ds_read_b64_tr_b16): in every 16-lane group, lane s points at 4 columns of key row
            //      s/4 and receives column s (of the group's 16) for the group's 4 key rows.  Column tile
            //      t is V columns t*32 .. t*32+31 in lane order.
            typedef short v4s_t __attribute__((ext_vector_type(4)));
            asm volatile("" : "+v"(v_at));
            constexpr int kVG = Cfg::kMT < 4 ? Cfg::kMT : 4;         // column tiles whose operands are read together
            constexpr int kVSteps = 2 * H * Cfg::kMT / kVG;
            u32x4_t va[2][kVG];
            auto read_v = [&](int step) {
                const int ks = step / (Cfg::kMT / kVG), t0 = step % (Cfg::kMT / kVG) * kVG;
#pragma unroll
                for (int u = 0; u < kVG; ++u) {
                    if (PART && (t0 + u) * 32 >= hd) continue;
#pragma unroll
                    for (int hv = 0; hv < 2; ++hv) {
                        const v4s_t r4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (__attribute__((address_space(3))) v4s_t *)(uintptr_t)((v_at ^ (uint32_t)((t0 + u) << 6)) + (16 * ks + 8 * hv) * Cfg::kRowBytes));
                        const uint2 r2 = __builtin_bit_cast(uint2, r4);
                        va[step & 1][u][2 * hv] = r2.x;
                        va[step & 1][u][2 * hv + 1] = r2.y;
                    }
                }
            };
            read_v(0);
#pragma unroll
            for (int step = 0; step < kVSteps; ++step) {
                const int ks = step / (Cfg::kMT / kVG), t0 = step % (Cfg::kMT / kVG) * kVG;
                if (step + 1 < kVSteps) read_v(step + 1);
#pragma unroll
                for (int u = 0; u < kVG; ++u) {
                    if (PART && (t0 + u) * 32 >= hd) continue;
                    o_acc[t0 + u] = mfma32<T>(va[step & 1][u], pk[ks >> 1][ks & 1], o_acc[t0 + u]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
        };
        if (live == 2) products(std::integral_constant<int, 2>{});
        if (kHalves && live == 1) products(std::integral_constant<int, 1>{});
        k_at ^= Cfg::kTileBytes;
        if (Cfg::kVBufs == 2) v_at ^= Cfg::kTileBytes;
        v_here[0] = next.v[0], v_here[1] = next.v[1];
        advance(next);
        tiles_landed();
        barrier();
    }

    // ---- epilogue: O^T / l, store.  Register r of column tile t is V column
    //      t*32 + 8*(r/4) + 4*lh + r%4 of query row ln: four consecutive columns per (t, r/4).
    l_run = halves_sum(l_run);
    const float inv = (l_run > 0.f) ? 1.f / l_run : 0.f;
    if (!whole) {
        // one of several ranges of the unit: normalised fp32 partial and base-2 LSE for the combine
        const TileRow row = my_row(this_lane());
        if (row.ok) {
            float *part_row = p.o_partial + part_of(row) * D;
#pragma unroll
            for (int t = 0; t < Cfg::kMT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<float4 *>(part_row + t * 32 + 8 * j + 4 * lh) =
                        make_float4(o_acc[t][4 * j] * inv, o_acc[t][4 * j + 1] * inv, o_acc[t][4 * j + 2] * inv,
                                    o_acc[t][4 * j + 3] * inv);
            if (lh == 0) p.lse_partial[part_of(row)] = (l_run > 0.f) ? m_run + fast_log2(l_run) : -INFINITY;
        }
        return;
    }
    const TileRow my = my_row(this_lane());
    if (my.ok && lh == 0) *lse_of(my) = (l_run > 0.f) ? (m_run + fast_log2(l_run)) * kLn2 : INFINITY;
    // The lane owns 8-byte pieces of its row, 16 of them: stored as they are, one instruction would touch
    // 32 rows of the output.  The wave's 32 x D tile goes through LDS instead (the V tiles are free
    // after the last barrier of the loop; each wave uses its own part, so no workgroup barrier) and
    // leaves as whole rows, 16 bytes per lane.
    constexpr int kStageRow = D * 2 + 16;                      // padded: the 8-byte writes of a column spread over the banks
    static_assert(4 * 32 * kStageRow <= (2 + Cfg::kVBufs) * Cfg::kTileBytes, "staging tile must fit the tiles");
    uint8_t *stage = &lds.k[0][0] + wave * (32 * kStageRow);
#pragma unroll
    for (int t = 0; t < Cfg::kMT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint2 o2;
            o2.x = pack2<T>(o_acc[t][4 * j] * inv, o_acc[t][4 * j + 1] * inv);
            o2.y = pack2<T>(o_acc[t][4 * j + 2] * inv, o_acc[t][4 * j + 3] * inv);
            *reinterpret_cast<uint2 *>(stage + ln * kStageRow + (t * 32 + 8 * j + 4 * lh) * 2) = o2;
        }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int kLanesPerRow = D * 2 / 16;                   // lanes that cover one row with 16 bytes each
    constexpr int kStageRows = 64 / kLanesPerRow;              // rows a wave stores per instruction
    const int piece = lane % kLanesPerRow;
#pragma unroll
    for (int r0 = 0; r0 < 32; r0 += kStageRows) {
        const int rr = r0 + lane / kLanesPerRow;               // row of the wave's tile
        const TileRow row = tile_row(wave * 32 + rr);
        if (row.ok && (!PART || piece * 8 < hd)) {
            uint16_t *dst = reinterpret_cast<uint16_t *>(p.out) + (int64_t)b * p.o_stride_b + (int64_t)row.head * p.o_stride_h +
                            (int64_t)(q0 + row.pos) * p.o_stride_t;
            store16(dst + piece * 8, *reinterpret_cast<const u32x4_t *>(stage + rr * kStageRow + piece * 16));
        }
    }
}

template <typename T, int D, bool PAGED, bool SOFTCAP, bool EXT, bool PART>
__global__ void __launch_bounds__(256, prefill_wgs_resident(D, PART)) prefill_kernel(const PrefillParams p) {
    __shared__ __attribute__((aligned(2 * PrefillCfg<D>::kTileBytes))) PrefillTileLds<D> lds;
    prefill_block<T, D, PAGED, SOFTCAP, EXT, PART>(p, blockIdx.x, -1, lds);
}

// The same blocks for a launch whose live sequences are known on the device only (token-major batches whose
// short blocks went to the decode kernels: p.long_ids, p.list_state[0] of them).  A grid sized for every batch
// row would be mostly workgroups that find nothing to do, and dispatching those costs as much time as the live
// ones' work once the batch has many decode rows.  Here as many workgroups as the device holds take blocks from
// the ordered list until it ends: workgroup w (on XCD w % 8) takes the blocks congruent to w % 8, so that the heads
// of a unit still meet in one L2, through one counter per XCD (p.list_state[1 + x], zeroed by the kernel that
// wrote the list).  Every workgroup leaves when its counter passes the end of the list.
template <typename T, int D, bool SOFTCAP, bool PART>
__global__ void __launch_bounds__(256, prefill_wgs_resident(D, true)) prefill_list_kernel(const PrefillParams p) {
    __shared__ __attribute__((aligned(2 * PrefillCfg<D>::kTileBytes))) PrefillTileLds<D> lds;
    __shared__ int s_item;
    const int n_long = p.list_state[0];
    const int heads_per_unit = (p.pack > 1) ? 1 : p.group;
    const int64_t units8 = ((int64_t)n_long * max(p.nsplits, 1) * p.nheads_k + 7) / 8 * 8;
    const int64_t total = (int64_t)p.num_mb * units8 * heads_per_unit;     // a multiple of 8
    const int x = blockIdx.x & 7;
    for (;;) {
        __syncthreads();   // the last block's LDS tiles and s_item are free
        if (threadIdx.x == 0) s_item = atomicAdd(&p.list_state[1 + x], 1);
        __syncthreads();
        const int64_t bid = (int64_t)__builtin_amdgcn_readfirstlane(s_item) * 8 + x;
        if (bid >= total) break;
        prefill_block<T, D, true, SOFTCAP, true, PART>(p, (unsigned)bid, n_long, lds);
    }
}

// Merge of the key ranges of token-major query blocks over a paged cache: one wave per (token, head).
// Partials are laid out (token, head, range): normalised fp32 rows and base-2 log-sum-exps, -inf for a
// range in which the row saw nothing.  out = sum_r e^{lse_r - LSE} O_r, LSE = log sum_r e^{lse_r}.
// grid: total_q * ceil(nheads / combine_heads) workgroups of 256 threads: the four waves take the heads of one token in turn,
// so what depends on the token alone (its sequence, the cut of that sequence's keys) is found once per workgroup and every
// early exit is taken by the whole workgroup.
// Bound by its chain of trips to memory (offsets -> lengths -> partials): with four heads per workgroup a wave merged one row
// per chain. 1024 tokens x 32 heads x 2 ranges, d = 128 (42 MB): 19.7 us with four heads per workgroup, 12.6 now.
template <typename T, int D>
__global__ void __launch_bounds__(256) prefill_combine_kernel(const PrefillParams p, const int heads_per_wg) {
    const int head_groups = (p.nheads + heads_per_wg - 1) / heads_per_wg;
    const int tok = blockIdx.x / head_groups;
    const int head0 = (blockIdx.x - tok * head_groups) * heads_per_wg;
    const int lane = threadIdx.x & 63;
    // the sequence of this token: last b with cu_seqlens_q[b] <= tok (empty sequences repeat an offset), counted by
    // the lanes side by side: one trip to memory where a bisection makes log2(batch) dependent ones
    int below = 0;
    for (int i = lane; i < p.batch; i += 64) below += (p.cu_seqlens_q[i] <= tok) ? 1 : 0;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) below += __shfl_xor(below, d, 64);
    const int b = __builtin_amdgcn_readfirstlane(max(below - 1, 0));
    const int Sq = p.cu_seqlens_q[b + 1] - p.cu_seqlens_q[b];
    const int Sk = min(p.seqused_k[b] + p.seqlen_k_add, p.max_blocks * p.page_size);
    if (Sq >= 1 && Sq <= p.skip_short) return;   // computed by the decode kernels (the whole workgroup: one token)
    const int longest = block_max_keys(p.seqused_k, p.batch, p.seqlen_k_add);
    int wl = p.window_left, wr = p.window_right;
    int norm_m = p.window_norm_m;
    if (norm_m <= 0 && (wl >= 0 || wr >= 0)) norm_m = longest;
    if (norm_m <= 0) norm_m = max(Sk, 1);
    normalize_window(wl, wr, p.causal, norm_m);
    const int sk = adaptive_split_keys(min(longest, p.max_blocks * p.page_size), p.nsplits);
    const KeyRanges kr = key_ranges(Sq, Sk, wl, wr, sk, p.nsplits);
    const int count = __builtin_amdgcn_readfirstlane(kr.count);
    if (count == 1) return;   // the tile that computed this row wrote it
    constexpr int C = D / 64;        // columns per lane
    constexpr int kTogether = 4;     // ranges whose rows are in flight together
#pragma unroll 2
    for (int head = head0 + (int)(threadIdx.x >> 6); head < min(head0 + heads_per_wg, p.nheads); head += 4) {
        const int64_t base = ((int64_t)tok * p.nheads + head) * p.nsplits;
        const float *rows = p.o_partial + base * D + lane * C, *lses = p.lse_partial + base;
        float mx = -INFINITY;
        for (int r = lane; r < count; r += 64) mx = fmaxf(mx, lses[r]);
        float v[kTogether][C];
        auto fetch = [&](int r0) {
#pragma unroll
            for (int i = 0; i < kTogether; ++i)
#pragma unroll
                for (int c = 0; c < C; ++c) v[i][c] = rows[(int64_t)min(r0 + i, count - 1) * D + c];
        };
        fetch(0);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d, 64));
        const float mx_use = (mx == -INFINITY) ? 0.f : mx;
        float acc[C];
#pragma unroll
        for (int c = 0; c < C; ++c) acc[c] = 0.f;
        float tot = 0.f;
        for (int r0 = 0; r0 < count; r0 += kTogether) {
            if (r0 > 0) fetch(r0);
#pragma unroll
            for (int i = 0; i < kTogether; ++i) {
                if (r0 + i >= count) break;
                const float w = fast_exp2(lses[r0 + i] - mx_use);
                tot += w;
#pragma unroll
                for (int c = 0; c < C; ++c) acc[c] += w * v[i][c];
            }
        }
        const float inv = (tot > 0.f) ? 1.f / tot : 0.f;
        uint16_t *dst = reinterpret_cast<uint16_t *>(p.out) + (int64_t)tok * p.o_stride_t + (int64_t)head * p.o_stride_h + lane * C;
        if (lane * C < p.headdim) {   // the partials are D wide; the output row ends at the head dimension
#pragma unroll
            for (int c = 0; c < C; ++c) dst[c] = from_float<T>(acc[c] * inv);
        }
        if (lane == 0) p.lse[(int64_t)head * p.lse_stride_h + tok] = (tot > 0.f) ? (mx + fast_log2(tot)) * kLn2 : INFINITY;
    }
}

static_assert(kBM == kPrefillTileRows, "the planning rules in fa_kernels.h assume this tile height");

template <typename T, int D> static hipError_t launch_prefill_d(const PrefillParams &p_in, hipStream_t stream) {
    PrefillParams p = p_in;
    const PrefillTiles tiles = prefill_tiling(p.group, p.nheads, p.max_seqlen_q, p.total_q, D, p.num_cus, p.causal && p.nsplits <= 1 && !p.long_ids);
    p.pack = tiles.pack;
    p.mb_run = tiles.mb_run;
    p.num_mb = tiles.num_mb;
    if (p.nsplits > 1 && (!p.block_table || !p.o_partial || !p.lse_partial)) return hipErrorInvalidValue;
    const int64_t units = (int64_t)p.batch * max(p.nsplits, 1) * p.nheads_k;
    p.units8 = (int32_t)((units + 7) / 8 * 8);
    const int64_t wgs = (int64_t)p.num_mb * p.units8 * (p.pack > 1 ? 1 : p.group);
    if (wgs <= 0 || wgs >= (1ll << 31)) return hipErrorInvalidValue;
    dim3 grid((unsigned)wgs);
    dim3 block(256);
    const bool softcap = p.softcap_post != 0.f;
    const bool paged = p.block_table != nullptr;
    p.pack_short = p.cu_seqlens_q ? prefill_pack_short(p.group, p.max_seqlen_q, p.total_q, p.batch) : 0;
    if (p.headdim > D || p.headdim < 8 || p.headdim % 8 != 0) return hipErrorInvalidValue;
    const bool part = p.headdim < D;
    // a head dimension below the compiled width always takes the kernels with every extension compiled in
    const bool ext = part || p.pack > 1 || p.nsplits > 1 || p.pack_short || p.skip_short > 0;
    if (p.long_ids) {
        // live sequences listed on the device: workgroups that stay and take blocks from the list
        if (!paged || !p.list_state || p.list_wgs <= 0 || !p.cu_seqlens_q) return hipErrorInvalidValue;
        dim3 lgrid((unsigned)std::min<int64_t>(p.list_wgs, wgs));
        if (softcap) {
            if (part)
                hipLaunchKernelGGL((prefill_list_kernel<T, D, true, true>), lgrid, block, 0, stream, p);
            else
                hipLaunchKernelGGL((prefill_list_kernel<T, D, true, false>), lgrid, block, 0, stream, p);
        } else {
            if (part)
                hipLaunchKernelGGL((prefill_list_kernel<T, D, false, true>), lgrid, block, 0, stream, p);
            else
                hipLaunchKernelGGL((prefill_list_kernel<T, D, false, false>), lgrid, block, 0, stream, p);
        }
        return hipGetLastError();
    }
    auto launch = [&](auto paged_c, auto softcap_c, auto ext_c) {
        constexpr bool kExt = decltype(ext_c)::value;
        if constexpr (kExt) {
            if (part) {
                hipLaunchKernelGGL((prefill_kernel<T, D, decltype(paged_c)::value, decltype(softcap_c)::value, true, true>), grid, block,
                                   0, stream, p);
                return;
            }
        }
        hipLaunchKernelGGL((prefill_kernel<T, D, decltype(paged_c)::value, decltype(softcap_c)::value, kExt, false>), grid, block, 0,
                           stream, p);
    };
    auto pick_ext = [&](auto paged_c, auto softcap_c) {
        if (ext) launch(paged_c, softcap_c, std::true_type{}); else launch(paged_c, softcap_c, std::false_type{});
    };
    auto pick_softcap = [&](auto paged_c) {
        if (softcap) pick_ext(paged_c, std::true_type{}); else pick_ext(paged_c, std::false_type{});
    };
    if (paged) pick_softcap(std::true_type{}); else pick_softcap(std::false_type{});
    return hipGetLastError();
}

template <typename T> static hipError_t launch_prefill_t(const PrefillParams &p, int headdim, hipStream_t stream) {
    switch (headdim) {
        case 64: return launch_prefill_d<T, 64>(p, stream);
        case 128: return launch_prefill_d<T, 128>(p, stream);
        case 256: return launch_prefill_d<T, 256>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

template <typename T> static hipError_t launch_prefill_combine_t(const PrefillParams &p, int headdim, hipStream_t stream) {
    // heads per workgroup: as many as leave eight workgroups per compute unit
    int heads = 4;
    while (heads < p.nheads && (int64_t)p.total_q * ((p.nheads + 2 * heads - 1) / (2 * heads)) >= 8ll * p.num_cus) heads *= 2;
    const int64_t wgs = (int64_t)p.total_q * ((p.nheads + heads - 1) / heads);
    if (wgs <= 0 || wgs >= (1ll << 31)) return hipErrorInvalidValue;
    dim3 grid((unsigned)wgs), block(256);
    switch (headdim) {
        case 64: hipLaunchKernelGGL((prefill_combine_kernel<T, 64>), grid, block, 0, stream, p, heads); break;
        case 128: hipLaunchKernelGGL((prefill_combine_kernel<T, 128>), grid, block, 0, stream, p, heads); break;
        case 256: hipLaunchKernelGGL((prefill_combine_kernel<T, 256>), grid, block, 0, stream, p, heads); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_prefill_combine(const PrefillParams &p, int dtype, int headdim, hipStream_t stream) {
    if (p.nsplits <= 1 || p.total_q <= 0) return hipSuccess;
    if (!p.cu_seqlens_q || !p.block_table || !p.o_partial || !p.lse_partial) return hipErrorInvalidValue;
    return dtype == 0 ? launch_prefill_combine_t<BF16>(p, headdim, stream) : launch_prefill_combine_t<FP16>(p, headdim, stream);
}

hipError_t launch_prefill(const PrefillParams &p, int dtype, int headdim, hipStream_t stream) {
    if (p.max_seqlen_q <= 0 || p.batch <= 0) return hipSuccess;
    return dtype == 0 ? launch_prefill_t<BF16>(p, headdim, stream) : launch_prefill_t<FP16>(p, headdim, stream);
}

}  // namespace fa
