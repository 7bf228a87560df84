// Sparse (QSA) attention over selection bodies: the kernel behind fnkv_attn_sparse, fnkv_qsa_attend / fnkv_attend and
// fnkv_qsp_attend (sparse.hip, qsa.hip and qsp.hip check the calls and plan the launches).
//
// What it computes (the reference's decode attention over a selected-block body, fn/kernels/qsa/attend.h:8-34,
// attend.cu:405-421, and its prompt form, qsa_prompt_attn.cu:229-436): row z of a launch sits at position q = depth + z
// and attends to the cells of its body's K = min((q + 1) / 4, 512) ascending 4-cell blocks and to its tail cells
// 4 ((q + 1) / 4) .. q, with the decoded Q8_0 / KV8 cells, fp32 scores, softmax statistics and accumulators. Block IDs
// outside the row's whole blocks, and an ID equal to the one before it, are ignored. A row that selects a block of an
// unmapped page (a slot trimmed under a captured launch, outside the contract) gets no output.
//
// How (MI355X):
//   * The pool's tiles hold 32 cells, a selection picks 4-cell blocks: where a selection scatters, reading whole tiles
//     moves (and computes) up to eight times the cells it asks for. Here eight selected blocks, in the body's order, make
//     a virtual tile: the tile layout (layout.h) keeps a block's K as 16 pieces of 64 contiguous bytes and its V as 8
//     of 256, so each lane loads its own operand bytes from its own block straight into the registers that
//     v_mfma_f32_16x16x32_f16 reads (K: 8 loads of 16 B; V: 16 of 12 B, of which 8 are its cells'), and the scores, the
//     softmax and PV run on the virtual tile as on a stored one. Entry e of the body is cell group e of virtual tile
//     e / 8, so no workgroup builds a list: a lane's block is one body word and one page-table word.
//   * A workgroup of 4 waves (one a SIMD; two workgroups a CU for prompt rows) owns (row, up to 16 query heads of a KV
//     head, split): wave w of split s takes virtual tiles 4 s + w, + 4 n_splits, ... Decode rows launch enough splits for
//     one tile a wave (at most 17 splits of a row's 65 tiles) where those are at most one workgroup a CU; prompt rows split
//     only while the rows alone do not fill the device, and a row of one split is finished here, without partials or a
//     merge.
//   * A tile's K and scales are requested while the previous tile is in its softmax and PV, its V while the next
//     scores run; every block of the wave's tiles is resolved (body word, then page) before the first.
//   * The workgroups are laid out so that an XCD's share of them is consecutive rows: a prompt's neighbouring rows
//     select much the same blocks and find them in that XCD's L2.
// What bounds it: decode rows, latency (depth word, body, page table, blocks, then the fold and the merge launch);
// prompt rows, VALU issue (the loop: about 455 instructions and 52 MFMAs a virtual tile, 84 more where it moves the
// softmax reference; with the rest of the kernel 619 and 52.5, issued in 76% of the cycles that a SIMD holds two waves; the
// blocks come from L2 at about 10 TB/s).
// Measured against a kernel that rebuilt each row's tile list in LDS and read whole tiles (kernel trace, us; 12 heads
// on one KV head unless said): 1,000 prompt rows at 40,000 cells 128.6 + no merge (1,398 in two chunks + 198 of
// merges); attn::attend rows at 196,608 cells, 3 rows 12.4 + 4.9 merge (20.5 + 6.1); 16 heads on 2 KV heads, one KV8
// row at 9,001 cells 8.4 + 4.1 (14.1 + 4.1); 48 heads, 5 clustered rows at 60,000 cells 12.5 + 4.9 (37.8 + 5.6); a row
// of 130 cells 8.5 + 4.0 (12.3 + 4.5).
#include "../../include/fnkv.h"
#include "common.h"
#include "decode_common.h"
#include "gather.h"
#include "layout.h"
#include "mfma.h"
#include "q8_0.h"
#include "rope.h"

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>

namespace fnkv {

namespace {

constexpr int32_t kW = kGatherWaves;
constexpr int32_t kGatherOS = kHeadDim + 4;                       // floats a row of a wave's fold buffer
constexpr int32_t kGatherSlot = (16 * kGatherOS + 16 * 2) * 4;    // a wave's 16 rows of values, then their (m, l)
constexpr int32_t kGatherQ = kW * kGatherSlot;                    // then the query operands: [block][lane] 16 B
constexpr int32_t kGatherQBytes = kBlocks * 64 * 16;              // (QLO: their low parts after them)
constexpr int32_t gather_lds(bool qlo) { return kGatherQ + (qlo ? 2 : 1) * kGatherQBytes + 64; }
static_assert(2 * gather_lds(false) <= 160 * 1024, "two workgroups a CU");
constexpr int32_t kMaxTiles = (kSelTopBlocks + 1 + 7) / 8;        // virtual tiles a row: 65
constexpr int32_t kMaxRegs = ((kMaxTiles + kW - 1) / kW + 7) / 8; // 8 tiles' entries a register: 3
constexpr int32_t kTileKib = kTileBytes / 1024;                   // 17
constexpr int32_t kPageKib = static_cast<int32_t>(kPageBlock / 1024);
static_assert(kTileBytes % 1024 == 0 && kPageBlock % 1024 == 0, "tiles sit at whole KiB");

typedef uint32_t u32x3a __attribute__((ext_vector_type(3), aligned(4)));

// 12 bytes at a 4-byte aligned address
__device__ __forceinline__ u32x3a load12(const uint8_t * p) { return *reinterpret_cast<const u32x3a *>(p); }

// a virtual tile's operands as this lane holds them
struct gather_regs {
    u32x4 k[8];      // [half][chunk]: 16 values of the lane's token (as a stored tile's chunk)
    u32x3a v[8][2];  // [chunk][half]: word 0 the lane's 4 cells of MFMA tile 2 chunk, word 2 of 2 chunk + 1
    u32x4 ks;        // lanes 0 .. 31: token lane's K scales
    u32x2 vs;        // (group lane / 16, block lane / 2 % 8, half lane % 2): its 4 cells' V scales
};

// S^T = K Q^T of a virtual tile, K codes in registers: out[h][r] is the score (q . k, unscaled) of token 16 h + 4 qg + r
// against row j
template <bool KV8, typename QOP, typename QLOP>
__device__ __forceinline__ void gather_scores(const u32x4 (&kw)[8], const uint8_t * sc, const QOP & qop, half8 sig,
                                              int32_t j, int32_t qg, floatx4 (&out)[2], const QLOP & qlo) {
    constexpr bool QLO = has_qlo<QLOP>;
    const half8 zero8 = {};
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    // chunk c's products (blocks 2 (c & 3), + 1 of half c / 4); KV8: one for its 64-value group. A chunk's scale FMAs
    // run one chunk behind its MFMAs, under the next chunk's
    floatx4 t[2][2];
    auto products = [&](int c) {
#pragma unroll
        for (int bb = 0; bb < 2; ++bb) {
            const int b = 2 * (c & 3) + bb;
            const half8 ka = widen8<QLO>(kw[c][2 * bb], kw[c][2 * bb + 1]);
            floatx4 & o = t[c & 1][KV8 ? 0 : bb];
            o = mfma16(ka, qop(b), KV8 && bb == 1 ? o : zero4);
            if constexpr (QLO) {
                o = mfma16(ka, qlo(b), o);
            }
        }
    };
    products(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        half8 ks[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ks[r] = *reinterpret_cast<const half8 *>(sc + (16 * h + 4 * qg + r) * 16);
        }
        floatx4 acc_s = zero4;
        if constexpr (!QLO) { // the 1152 bias of the widened codes, taken out through the scores' start
            const half8 srow = qg < 2 ? *reinterpret_cast<const half8 *>(sc + (16 * h + j) * 16) : zero8;
            acc_s = mfma16(srow, sig, zero4) * -1152.0f;
        }
#pragma unroll
        for (int ld = 0; ld < 4; ++ld) {
            const int c = 4 * h + ld;
            if (c + 1 < 8) {
                products(c + 1);
            }
#pragma unroll
            for (int bb = 0; bb < (KV8 ? 1 : 2); ++bb) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    acc_s[r] = __builtin_fmaf(static_cast<float>(ks[r][2 * ld + bb]), t[c & 1][bb][r], acc_s[r]);
                }
            }
            __asm__ volatile("" : "+v"(acc_s)); // pin the chunk's FMAs: two chunks' results live at a time
            __builtin_amdgcn_sched_barrier(0);
        }
        out[h] = acc_s;
    }
}

// The row's new cells that this workgroup reads (bit c: cell depth + c) or owns: quantized and written before its
// block loads (several workgroups may write one cell: the same bytes; a cell of an unmapped page is not written).
// Prepared rows (fp): K = the F32 RMS norm and IMROPE of kv_k's row c (the row's own cell z from own_x / own_g, loaded
// early, at the pairs' angles rp), V = kv_v's row c; else one row's k_new / v_new.
__device__ __forceinline__ void gather_append(const gather_args & a, int32_t kvh, int32_t z, int64_t depth,
                                              uint32_t cells, bool own, const rope_pairs & rp,
                                              float4 own_x, float4 own_g, int32_t wave, int32_t lane) {
    const pool_view & pv = a.pv;
    for (int32_t job = wave; job < 2 * (z + 1); job += kW) {
        const int32_t c = job >> 1, kv = job & 1;
        if (((cells >> c) & 1u) == 0) {
            continue;
        }
        const int64_t pos = depth + c;
        const int64_t src = (int64_t(c) * pv.h_kv + kvh) * kHeadDim;
        float x[4];
        if (a.fp.qfull == nullptr) {
            if (a.new_f32) {
                load4<true>(static_cast<const float *>(kv ? a.v_new : a.k_new) + src, lane, x);
            } else {
                load4<false>(static_cast<const uint16_t *>(kv ? a.v_new : a.k_new) + src, lane, x);
            }
        } else if (kv == 0) {
            if (c == z) {
                norm_rope_apply(x, own_x, own_g, rp, lane);
            } else {
                norm_rope(x, a.fp.kv_k + src, a.fp.k_norm, a.fp.pos, a.fp.rows, c, a.fp.theta_scale, lane);
            }
            if (own && c == z && a.fp.k_f32 != nullptr) {
                reinterpret_cast<float4 *>(a.fp.k_f32 + src)[lane] = make_float4(x[0], x[1], x[2], x[3]);
            }
        } else if (c == z) {
            x[0] = own_x.x;
            x[1] = own_x.y;
            x[2] = own_x.z;
            x[3] = own_x.w;
        } else {
            load4<true>(a.fp.kv_v + src, lane, x);
        }
        if (__builtin_expect(page_mapped(a.table, pos), 1)) {
            quantize_store_fmt(x, lane, tile_of(pv, a.table, a.layer, kvh, pos), static_cast<int32_t>(pos & 31), kv,
                               pv.format);
        }
    }
}

// KV8: the pool's group-64 format. QLO: q as fp16 hi + lo, exact codes and 6 more bits of P (the attn::attend calls).
// MANY: a wave may take several tiles (prompt rows, and decode rows of many KV heads); else at most one. Two workgroups a
// CU fit the LDS without QLO, and the registers of MANY.
template <bool KV8, bool QLO, bool MANY>
__global__ __launch_bounds__(64 * kW, MANY && !QLO ? 2 : 1) void gather_kernel(gather_args a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int32_t lane = static_cast<int32_t>(threadIdx.x) & 63;
    const int32_t wave = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(threadIdx.x) >> 6);
    const int32_t j = lane & 15, qg = lane >> 4;
    // workgroup -> (row, head tile, split): workgroups go to the 8 XCDs in turn, so XCD x takes items
    // x total / 8 .. of the row-major list
    int32_t item;
    {
        const int32_t total = static_cast<int32_t>(gridDim.x), lin = static_cast<int32_t>(blockIdx.x);
        const int32_t per = total >> 3, rem = total & 7, x = lin & 7;
        item = x * per + (x < rem ? x : rem) + (lin >> 3);
    }
    const int32_t split = item % a.n_splits;
    item /= a.n_splits;
    const int32_t head_tile = item % (a.pv.h_kv * a.head_tiles), z = item / (a.pv.h_kv * a.head_tiles);
    const int32_t kvh = head_tile / a.head_tiles, rt = head_tile % a.head_tiles;
    const int32_t G_t = a.G - 16 * rt < 16 ? a.G - 16 * rt : 16; // this workgroup's query heads
    const int32_t head0 = kvh * a.G + 16 * rt;                   // the first of them
    const bool prep = a.fp.qfull != nullptr;

    // A launch that prepares its rows: the inputs are requested first (wave w takes heads w, w + 4, ...; a head past
    // the last takes the last and is not used). Unset otherwise (never read).
    float4 xq[4], gq, own_x, own_g;
    int32_t pq;
    {
        const float u = __builtin_nondeterministic_value(0.0f);
        xq[0] = xq[1] = xq[2] = xq[3] = gq = own_x = own_g = make_float4(u, u, u, u);
        pq = __builtin_nondeterministic_value(0);
    }
    if (prep) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t h = wave + kW * i < G_t ? wave + kW * i : G_t - 1;
            xq[i] = reinterpret_cast<const float4 *>(a.fp.qfull + (int64_t(z) * a.hq + head0 + h) * 512)[lane];
        }
        gq = reinterpret_cast<const float4 *>(a.fp.q_norm)[lane];
        if (a.fp.kv_k != nullptr) {
            const int64_t crow = (int64_t(z) * a.pv.h_kv + kvh) * kHeadDim;
            own_x = reinterpret_cast<const float4 *>((wave == (2 * z + 1) % kW ? a.fp.kv_v : a.fp.kv_k) + crow)[lane];
            own_g = reinterpret_cast<const float4 *>(a.fp.k_norm)[lane];
        }
        // the row's rope position on the lane's plane: [plane][row], [row][plane], or the text position on every plane
        pq = a.fp.pos == nullptr ? a.fp.pos0 + z
             : a.fp.row_major    ? a.fp.pos[4 * z + rope_plane(lane)]
                                 : rope_pos(a.fp.pos, a.fp.rows, z, lane);
    }
    int64_t depth = a.depth;
    if (a.depth_dev != nullptr) {
        depth = *a.depth_dev;
        if (depth < 0 || depth + a.T > a.cap) { // refused: nothing is written; one workgroup reports it
            if (blockIdx.x == 0 && threadIdx.x == 0) {
                atomicOr(a.err, FNKV_DEV_ERR_DEPTH);
            }
            return;
        }
    }
    const int32_t q = static_cast<int32_t>(depth) + z; // at most kSelMaxCells
    const sel_shape sel(q);
    if (kW * split >= sel.tiles) {
        return; // past the row's tiles (the merge reads only the splits that hold some)
    }
    // the row's body
    int64_t words = 0;
    if (a.offsets != nullptr) { // a prompt row: its slab, then its offset in the slab
        const int32_t slab = z / kSlabRows;
        words = int64_t(slab) * kSlabWords + a.offsets[slab * (kSlabRows + 1) + z % kSlabRows] / 4;
    } else { // the earlier rows' words come first
        for (int32_t t = 0; t < z; ++t) {
            const sel_shape s(static_cast<int32_t>(depth) + t);
            words += 2 + s.K + s.tail;
        }
    }
    const uint32_t * const body = a.body + words + 2;

    // Every entry of this wave's tiles: register m, lane l holds entry l % 8 of the wave's tile 8 m + l / 8. First the
    // body's words, then the page-table words.
    constexpr int32_t M = MANY ? kMaxRegs : 1;
    int32_t word[M], before[M];
#pragma unroll
    for (int32_t m = 0; m < M; ++m) {
        const int32_t e = 8 * (kW * (split + a.n_splits * (8 * m + (lane >> 3))) + wave) + (lane & 7);
        const bool in = (MANY || lane < 8) && e < sel.K;
        word[m] = in ? static_cast<int32_t>(body[e]) : -1;
        before[m] = in && e > 0 ? static_cast<int32_t>(body[e - 1]) : -1;
    }
    rope_pairs rp = {};
    if (prep) { // the row's rope angle while the body's words are in flight
        int32_t p = pq;
        __asm__ volatile("" : "+v"(p)); // the position's load is waited for here, not where it was issued
        float sn, cs;
        rope_angle(sn, cs, p, a.fp.theta_scale, lane);
        rp = rope_pairs_of(sn, cs, lane);
    }

    int32_t id[M], page[M];
    bool good[M];
#pragma unroll
    for (int32_t m = 0; m < M; ++m) {
        const int32_t e = 8 * (kW * (split + a.n_splits * (8 * m + (lane >> 3))) + wave) + (lane & 7);
        const bool is_tail = (MANY || lane < 8) && e == sel.K && sel.tail != 0;
        good[m] = is_tail || (word[m] >= 0 && word[m] < sel.n_vis && word[m] != before[m]);
        id[m] = !good[m] ? 0 : is_tail ? sel.n_vis : word[m];
        page[m] = a.table[id[m] >> 6]; // 4-cell block -> page of 256 cells
    }
    // the query operands in LDS: operand (block b, lane (row j, qg)) is row j's values 32 b + 8 qg .. + 7, rows past the
    // heads zero (or the last head's: computed and never written)
    uint8_t * const qlds = smem + kGatherQ;
    if (prep) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t h = wave + kW * i;
            float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (h < G_t) {
                norm_rope_apply(y, xq[i], gq, rp, lane);
                if (split == 0 && a.fp.q_f32 != nullptr) {
                    reinterpret_cast<float4 *>(a.fp.q_f32 + (int64_t(z) * a.hq + head0 + h) * kHeadDim)[lane] =
                        make_float4(y[0], y[1], y[2], y[3]);
                }
            }
            // value 4 lane + i of head h is element 4 (lane & 1) + i of operand (block lane / 8, lane (h, (lane & 7) / 2))
            uint8_t * const at = qlds + ((lane >> 3) * 64 + ((lane & 7) >> 1) * 16 + h) * 16 + (lane & 1) * 8;
            *reinterpret_cast<uint2 *>(at) = pack4_f16(y, 1.0f);
            if constexpr (QLO) {
                float lo[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    lo[e] = y[e] - static_cast<float>(static_cast<_Float16>(y[e]));
                }
                *reinterpret_cast<uint2 *>(at + kGatherQBytes) = pack4_f16(lo, 1.0f);
            }
        }
    } else {
        const int64_t row = (int64_t(z) * a.hq + head0 + (j < G_t ? j : G_t - 1)) * kHeadDim + 8 * qg;
#pragma unroll
        for (int i = 0; i < kBlocks / kW; ++i) {
            const int32_t b = wave + kW * i;
            *reinterpret_cast<u32x4 *>(qlds + (b * 64 + lane) * 16) =
                *reinterpret_cast<const u32x4 *>(a.q + row + b * kQK);
            if constexpr (QLO) {
                *reinterpret_cast<u32x4 *>(qlds + kGatherQBytes + (b * 64 + lane) * 16) =
                    *reinterpret_cast<const u32x4 *>(a.q_lo + row + b * kQK);
            }
        }
    }
    // ... into the wave's own fold slot, past its scales: entry i's code (KiB offset of its tile in the (layer, head)
    // plane, 8 times, plus its block of the tile) and the cells of it to attend (4, the tail's, or none)
    uint8_t * const slot = smem + wave * kGatherSlot;
    uint32_t * const codes = reinterpret_cast<uint32_t *>(slot + 2048);
    uint8_t * const counts = slot + 2048 + 64 * kMaxRegs * 4;
    bool hole = false; // a selected block of an unmapped page: page 0 is read in its place, and the row gets no output
#pragma unroll
    for (int32_t m = 0; m < M; ++m) {
        const int32_t phys = page[m] >= 0 ? page[m] : 0;
        hole = hole || (good[m] && page[m] < 0);
        good[m] = good[m] && page[m] >= 0;
        const uint32_t kib = static_cast<uint32_t>(phys) * static_cast<uint32_t>(a.pv.h_kv * kPageKib) +
                             static_cast<uint32_t>((id[m] >> 3) & 7) * kTileKib;
        codes[64 * m + lane] = kib * 8 + static_cast<uint32_t>(id[m] & 7);
        counts[64 * m + lane] = static_cast<uint8_t>(!good[m] ? 0 : id[m] == sel.n_vis ? sel.tail : 4);
    }

    // New cells (decode rows; the form of prompt rows has none): the ones whose block this workgroup reads, and the row's
    // own cell by its owner: the split that holds the tail entry, or split 0 when the row has no tail
    const bool writes = (!MANY || QLO) && (a.k_new != nullptr || a.fp.kv_k != nullptr);
    uint32_t * const seen = reinterpret_cast<uint32_t *>(smem + gather_lds(QLO) - 64); // a word a wave
    if (writes) {
        uint32_t mine = 0;
        for (int32_t c = 0; c <= z; ++c) {
            bool hit = false;
#pragma unroll
            for (int32_t m = 0; m < M; ++m) {
                hit = hit || (good[m] && id[m] == static_cast<int32_t>((depth + c) >> 2));
            }
            mine |= __any(hit) ? 1u << c : 0u;
        }
        if (lane == 0) {
            seen[wave] = mine;
        }
    }
    barrier_keep_loads(); // the query operands and `seen` are in LDS
    if (writes) {
        uint32_t cells = 0;
#pragma unroll
        for (int w = 0; w < kW; ++w) {
            cells |= seen[w];
        }
        int32_t owner = sel.tail != 0 ? (sel.K >> 3) / kW : 0;
        if constexpr (MANY) {
            owner %= a.n_splits;
        }
        const bool own = rt == 0 && owner == split;
        cells |= own ? 1u << z : 0u;
        if (cells != 0) { // uniform in the workgroup
            gather_append(a, kvh, z, depth, cells, own, rp, own_x, own_g, wave, lane);
            __syncthreads(); // the stores are done (workgroup scope) before any wave loads a block
        }
    }

    const uint8_t * const base = a.pv.base + int64_t(a.layer) * a.pv.layer_stride + int64_t(kvh) * kPageBlock;
    auto tile_base = [base](uint32_t c) { return base + int64_t(c >> 3) * 1024; };
    gather_regs g;
    auto load_k = [&](int32_t t) {
        const uint32_t cks = codes[8 * t + ((lane >> 2) & 7)];
        const uint32_t cvs = codes[8 * t + 4 * (lane & 1) + qg];
        g.ks = *reinterpret_cast<const u32x4 *>(tile_base(cks) + kKScales + (4 * (cks & 7) + (lane & 3)) * 16);
        g.vs = *reinterpret_cast<const u32x2 *>(tile_base(cvs) + kVScales + (cvs & 3) * 128 + ((lane >> 1) & 7) * 16 +
                                                ((cvs >> 2) & 1) * 8);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t c = codes[8 * t + 4 * h + (j >> 2)];
            const uint8_t * p =
                tile_base(c) + ((c >> 2) & 1) * 4096 + (16 * qg + 4 * static_cast<int32_t>(c & 3) + (j & 3)) * 16;
#pragma unroll
            for (int ld = 0; ld < 4; ++ld) {
                g.k[4 * h + ld] = *reinterpret_cast<const u32x4 *>(p + ld * 1024);
            }
        }
    };
    auto load_v = [&](int32_t t) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t c = codes[8 * t + 4 * h + qg];
            // (from the middle chunk: all eight lie within a load's immediate offset)
            const uint8_t * p =
                tile_base(c) + kVCodes + 4096 + (16 * static_cast<int32_t>(c & 3) + j) * 16 + ((c >> 2) & 1) * 4;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                g.v[b][h] = load12(p + (b - 4) * 1024);
            }
        }
    };
    // the wave's tiles (uniform)
    const int32_t first = kW * split + wave;
    const int32_t n_w = __builtin_amdgcn_readfirstlane(
        sel.tiles > first ? (sel.tiles - first + kW * a.n_splits - 1) / (kW * a.n_splits) : 0);
    if (n_w > 0) {
        load_k(0);
        load_v(0);
    }

    auto q_at = [&](int b) { return *reinterpret_cast<const half8 *>(qlds + (b * 64 + lane) * 16); };
    auto qlo_at = [&](int b) { return *reinterpret_cast<const half8 *>(qlds + kGatherQBytes + (b * 64 + lane) * 16); };
    half8 sig = {}; // QLO: the codes enter exactly, no bias operand
    if constexpr (!QLO) {
        half8 qop[kBlocks];
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
            qop[b] = q_at(b);
        }
        sig = q_sums(qop, qg);
    }

    floatx4 acc[16];
    floatx4 lv = {0.0f, 0.0f, 0.0f, 0.0f}; // sum_t P[t][row] s_v[t][b]: lane (row j, qg) holds b = 4 qg + r
    float m_run = __any(hole) ? __builtin_nanf("") : kNegInf; // (a NaN stays one: the folds write nothing then)
    float l_run = 0.0f;
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        acc[m] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const half8 zero8 = {};
    for (int32_t t = 0; t < n_w; ++t) {
        uint8_t * const scales = slot + (t & 1) * 1024; // K [32][8], then V [4][8][8]; two tiles' in turn
        {
            // the scales into LDS; V scales of cells that are not attended become zero, whatever is stored there
            if (lane < 32) {
                *reinterpret_cast<u32x4 *>(scales + lane * 16) = g.ks;
            }
            const int32_t nv = counts[8 * t + 4 * (lane & 1) + qg];
            u32x2 v = g.vs;
            v[0] = nv >= 2 ? v[0] : nv == 1 ? v[0] & 0xffffu : 0u;
            v[1] = nv >= 4 ? v[1] : nv == 3 ? v[1] & 0xffffu : 0u;
            *reinterpret_cast<u32x2 *>(scales + 512 + lane * 8) = v;
        }
        floatx4 sc[2];
        if constexpr (QLO) {
            gather_scores<KV8>(g.k, scales, q_at, sig, j, qg, sc, qlo_at);
        } else {
            gather_scores<KV8>(g.k, scales, q_at, sig, j, qg, sc, no_qlo());
        }
        if (MANY && t + 1 < n_w) {
            load_k(t + 1);
        }
        float pf[8];
        {
            const int32_t n0 = counts[8 * t + qg], n1 = counts[8 * t + 4 + qg];
            float alpha;
            gather_softmax<QLO>(sc, n0, n1, a.c2, m_run, l_run, pf, alpha);
            if (MANY && __any(alpha != 1.0f)) { // (one tile: the accumulators are still zero)
#pragma unroll
                for (int m = 0; m < 16; ++m) {
                    acc[m] *= alpha;
                }
                lv *= alpha;
            }
        }
        half8 ph, pl;
        if constexpr (QLO) {
            ph = to_half8_rtz(pf);
        } else {
            split_hilo(pf, ph, pl);
            // A of the bias MFMAs: lane (block j < 8, qg): s_v of its group's 8 slots
            const half8 sva =
                j < 8 ? *reinterpret_cast<const half8 *>(scales + 512 + qg * 128 + j * 16) : zero8;
            lv = mfma16(sva, ph, lv);
            lv = mfma16(sva, pl, lv);
        }
        // two value blocks at a time: their hi terms, then their lo terms (an accumulator's two MFMAs four apart)
#pragma unroll
        for (int b0 = 0; b0 < 8; b0 += 2) {
            half8 hi[2], lo[2], va[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int b = b0 + i;
                if (KV8 && i == 1) { // block b shares block b - 1's scale
                    hi[1] = hi[0];
                    lo[1] = lo[0];
                } else {
                    const half8 vs = *reinterpret_cast<const half8 *>(scales + 512 + qg * 128 + b * 16);
                    if constexpr (QLO) {
                        scale_hilo<true>(pf, ph, vs, hi[i], lo[i]);
                    } else {
                        scale_hilo_pk(ph, pl, vs, hi[i], lo[i]);
                    }
                }
                va[i][0] = widen8<QLO>(g.v[b][0][0], g.v[b][1][0]);
                va[i][1] = widen8<QLO>(g.v[b][0][2], g.v[b][1][2]);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                acc[2 * b0 + m] = mfma16(va[m >> 1][m & 1], hi[m >> 1], acc[2 * b0 + m]);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                acc[2 * b0 + m] = mfma16(va[m >> 1][m & 1], lo[m >> 1], acc[2 * b0 + m]);
            }
            __builtin_amdgcn_sched_barrier(0); // two blocks' operands live at a time
        }
        if (MANY && t + 1 < n_w) {
            load_v(t + 1);
        }
    }
    // the V bias: acc[m] carries 1152 * lv[b = m / 2]; lv[b] of this lane's row sits in lane (j, b / 4), element b % 4
    if constexpr (!QLO) {
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
            const float lb = __shfl(lv[b & 3], j + 16 * (b >> 2));
            acc[2 * b] -= 1152.0f * lb;
            acc[2 * b + 1] -= 1152.0f * lb;
        }
    }
    l_run = rows_sum(l_run);

    // the gates of this wave's rows of the fold, requested before its barrier
    float4 gates[4] = {};
    if (a.n_splits == 1 && a.fin.gate != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t r = wave + kW * i < G_t ? wave + kW * i : G_t - 1;
            gates[i] = finish_gate(a.fin, int64_t(z) * a.hq + head0 + r, lane * 4);
        }
    }

    // ---- fold the waves in order: each writes its unscaled rows and (m, l) into its own slot, the reads scale ----
    float * const mine = reinterpret_cast<float *>(slot);
    if (j < G_t) {
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            *reinterpret_cast<floatx4 *>(mine + j * kGatherOS + 16 * m + 4 * qg) = acc[m];
        }
    }
    if (qg == 0) {
        *reinterpret_cast<float2 *>(mine + 16 * kGatherOS + 2 * j) = float2{m_run, l_run};
    }
    if (__builtin_expect(m_run != m_run, 0) && a.err != nullptr && lane == 0) {
        atomicOr(a.err, FNKV_DEV_ERR_DEPTH);
    }
    __syncthreads();
    // thread -> (row, 4 values): a wave a row, its 64 lanes the row's 256 values
    const int32_t c0 = lane * 4;
    const float * const slots = reinterpret_cast<const float *>(smem);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int32_t r = wave + kW * i;
        if (r >= G_t) {
            break;
        }
        float2 ml[kW];
        float Mr = kNegInf;
#pragma unroll
        for (int w = 0; w < kW; ++w) {
            ml[w] = *reinterpret_cast<const float2 *>(slots + w * (kGatherSlot / 4) + 16 * kGatherOS + 2 * r);
            Mr = __builtin_elementwise_maximum(Mr, ml[w].x); // (a NaN stays one)
        }
        const float Mu = Mr == kNegInf ? 0.0f : Mr;
        float L = 0.0f;
        floatx4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < kW; ++w) {
            const float f = __builtin_amdgcn_exp2f(ml[w].x - Mu);
            L = __builtin_fmaf(ml[w].y, f, L);
            const floatx4 v = *reinterpret_cast<const floatx4 *>(slots + w * (kGatherSlot / 4) + r * kGatherOS + c0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] = __builtin_fmaf(v[e], f, sum[e]);
            }
        }
        const int64_t row = int64_t(z) * a.hq + head0 + r;
        if (a.n_splits == 1) {
            if (__builtin_expect(Mr == Mr, 1)) { // (uniform: a wave a row)
                finish4(a.fin, row, c0, sum, L, gates[i]);
            }
        } else {
            const int64_t prow = ((int64_t(z) * a.n_splits + split) * a.pv.h_kv + kvh) * a.G + 16 * rt + r;
            *reinterpret_cast<floatx4 *>(a.po + prow * kHeadDim + c0) = sum;
            if (lane == 0) {
                *reinterpret_cast<float2 *>(a.pml + prow * 2) = float2{Mr, L};
            }
        }
    }
}

template <bool KV8, bool QLO, bool MANY> void set_gather_attr() {
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(gather_kernel<KV8, QLO, MANY>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, gather_lds(QLO));
}

template <bool KV8, bool QLO, bool MANY> void launch(uint32_t grid, const gather_args & a, hipStream_t st) {
    hipLaunchKernelGGL((gather_kernel<KV8, QLO, MANY>), dim3(grid), dim3(64 * kW), gather_lds(QLO), st, a);
}

} // namespace

void launch_gather(int32_t device, const gather_args & a, hipStream_t st) {
    static std::once_flag attr_once[64]; // once per device; a racing first caller waits for it
    if (device >= 0 && device < 64) {
        std::call_once(attr_once[device], [device]() {
            int32_t cur = 0;
            (void)hipGetDevice(&cur);
            (void)hipSetDevice(device);
            set_gather_attr<false, false, false>();
            set_gather_attr<true, false, false>();
            set_gather_attr<false, true, false>();
            set_gather_attr<true, true, false>();
            set_gather_attr<false, false, true>();
            set_gather_attr<true, false, true>();
            set_gather_attr<false, true, true>();
            set_gather_attr<true, true, true>();
            (void)hipGetLastError();
            (void)hipSetDevice(cur);
        });
    }
    const uint32_t grid =
        static_cast<uint32_t>(a.n_splits) * static_cast<uint32_t>(a.pv.h_kv * a.head_tiles) * static_cast<uint32_t>(a.T);
    const bool kv8 = a.pv.format == kFormatKV8;
    if (a.many && a.q_lo != nullptr) {
        kv8 ? launch<true, true, true>(grid, a, st) : launch<false, true, true>(grid, a, st);
    } else if (a.many) {
        kv8 ? launch<true, false, true>(grid, a, st) : launch<false, false, true>(grid, a, st);
    } else if (a.q_lo != nullptr) {
        kv8 ? launch<true, true, false>(grid, a, st) : launch<false, true, false>(grid, a, st);
    } else {
        kv8 ? launch<true, false, false>(grid, a, st) : launch<false, false, false>(grid, a, st);
    }
}

} // namespace fnkv
