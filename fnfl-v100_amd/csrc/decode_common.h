// Shared by the attention launches over the pool: the dense launch's arguments, its walk of a split's tiles and its
// append of the step's new cells (stream.hip), the split merge's arguments (decode.hip) and the sparse launches'
// entry (sparse.hip).
#pragma once

#include "../../include/fnkv.h"
#include "common.h"
#include "layout.h"
#include "mfma.h"
#include "q8_0.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace fnkv {

constexpr float kNegInf = -__builtin_inff();

struct dec_args {
    pool_view pv;
    const uint16_t * q; // fp16 [n_seq][T][hq][256]
    const void * k_new; // optional [n_seq][T][h_kv][256] fp16 / fp32: the step's new cells, appended by the launch
    const void * v_new;
    int32_t new_f32;
    float * po;         // [total_splits][h_kv][R][256] partial accumulators
    float * pml;        // [total_splits][h_kv][R][2] partial (m, l), base-2 domain
    float c2;           // scale * log2(e)
    int32_t layer, T, G, hq, R, n_seq, split_tokens;
    // dense: 1 when a sequence's n splits stride over its tiles (split j takes tiles j, j + n, ...; at most 128 a
    // split), 0 when split j takes the cells j split_tokens .. + split_tokens - 1
    int32_t strided;
    int32_t slot[FNKV_MAX_SEQS];
    // each sequence's context; with ctx_dev set, the host's bound on it instead (the launch's grid and workspace follow
    // from the bound, the work from the device word, so one captured launch serves every step up to the bound)
    int64_t ctx[FNKV_MAX_SEQS];
    int32_t split0[FNKV_MAX_SEQS + 1]; // first split of each sequence; split0[n_seq] = total
    const int64_t * ctx_dev = nullptr; // device contexts [n_seq], read by the launch; null: ctx[] are the contexts
    uint32_t * err = nullptr;          // with a device word: FNKV_DEV_ERR_DEPTH for a refused context (nothing written)
    // the split-K fold inside the launch (stream kernel, grid resident at once): fold state words (kFoldWords a
    // (sequence, KV head); zeroed before a workspace's first launch, each launch leaves them ready for the next), the
    // fp16 output, and the bound of every wait
    // (real-time ticks, 100 MHz). Null: the splits' partials go to the merge kernel.
    uint32_t * fold = nullptr;
    uint16_t * out = nullptr;
    int64_t fold_spin = 0;
#ifdef FNKV_TIMING
    uint64_t * ts; // per workgroup: 16 real-time stamps (instrumented builds only)
#endif
};
// fold state of a (sequence, KV head): the arrival counter, a spare word, and a state word per row; a launch adds
// kFoldEpoch to the counter in all (more than any pair's splits)
constexpr int32_t kFoldWords = 2 + FNKV_MAX_ROWS;
constexpr uint32_t kFoldEpoch = 1024;

#ifdef FNKV_TIMING
#define FNKV_STAMP(k)                                                                                                \
    do {                                                                                                             \
        if (a.ts != nullptr && threadIdx.x == 0) {                                                                   \
            a.ts[(blockIdx.y * gridDim.x + blockIdx.x) * 16 + (k)] = __builtin_amdgcn_s_memrealtime();                   \
            a.ts[(blockIdx.y * gridDim.x + blockIdx.x) * 16 + 7] =                                                       \
                (uint64_t(__builtin_amdgcn_s_getreg((15 << 11) | 20)) << 32) |                                           \
                uint64_t(__builtin_amdgcn_s_getreg((31 << 11) | 4));                                                     \
        }                                                                                                            \
        __builtin_amdgcn_s_waitcnt(0);                                                                               \
    } while (0)
#define FNKV_STAMP_WAVE()                                                                                            \
    do {                                                                                                             \
        if (a.ts != nullptr && (threadIdx.x & 63) == 0) {                                                            \
            a.ts[(blockIdx.y * gridDim.x + blockIdx.x) * 16 + 8 + (threadIdx.x >> 6)] =                              \
                __builtin_amdgcn_s_memrealtime();                                                                    \
        }                                                                                                            \
        __builtin_amdgcn_s_waitcnt(0);                                                                               \
    } while (0)
#endif
#if defined(FNKV_TIMING) && defined(FNKV_TIMING_PHASES)
// phase clocks of wave 0 (20-bit shader cycle counter, no memory counters touched), summed over the loop: a build of
// their own, since the clock reads constrain the loop's schedule (and its registers) more than the stamps do
#define FNKV_PHASE_DECL() uint32_t ph_last = 0, ph_sum[8] = {0, 0, 0, 0, 0, 0, 0, 0}
#define FNKV_PHASE(p)                                                                                                \
    do {                                                                                                             \
        const uint32_t now = static_cast<uint32_t>(__builtin_amdgcn_s_memtime());                                  \
        if ((p) > 0) {                                                                                               \
            ph_sum[(p)-1] += now - ph_last;                                                                          \
        }                                                                                                            \
        ph_last = now;                                                                                               \
    } while (0)
#define FNKV_PHASE_STORE()                                                                                           \
    do {                                                                                                             \
        if (a.ts != nullptr && threadIdx.x == 0) {                                                                   \
            for (int p_ = 0; p_ < 8; ++p_) {                                                                         \
                a.ts[4096 * 16 + (blockIdx.y * gridDim.x + blockIdx.x) * 8 + p_] = ph_sum[p_];                        \
            }                                                                                                        \
        }                                                                                                            \
    } while (0)
#else
#define FNKV_PHASE_DECL()                                                                                            \
    do {                                                                                                             \
    } while (0)
#define FNKV_PHASE(p)                                                                                                \
    do {                                                                                                             \
    } while (0)
#define FNKV_PHASE_STORE()                                                                                           \
    do {                                                                                                             \
    } while (0)
#endif
#ifndef FNKV_TIMING
#define FNKV_STAMP_WAVE()                                                                                            \
    do {                                                                                                             \
    } while (0)
#define FNKV_STAMP(k)                                                                                                \
    do {                                                                                                             \
    } while (0)
#endif

__device__ __forceinline__ int32_t seq_of(const dec_args & a, int32_t split);

// A lane's page-table entry, loaded by every lane (a lane past the walk reads entry 0; guard_unmapped replaces its
// value), so the load is not under a branch: there the compiler would first wait for every load issued before it
// (the launch's Q rows)
__device__ __forceinline__ int32_t page_of(const int32_t * table, bool active, int32_t idx) {
    return table[active ? idx : 0];
}

// The tiles a dense workgroup walks, at most 128 (splits of at most kMaxSplitPages pages): lane i holds the physical
// pages of walk tiles i and 64 + i, so a tile's page is a lane read.
constexpr int32_t kMaxSplitPages = 16;
struct split_src {
    int32_t n_tiles = 0;
    int32_t page_lane = 0, page_hi = 0;
    int32_t g0 = 0, stride = 1; // walk tile i is the sequence's tile g0 + stride i

    // The split's own cells b .. e, or (strided) split j of the sequence's n takes its tiles j, j + n, ...; the strided
    // page lookups are sized by the bound a.ctx[s], so they need not wait for a context read from the device
    __device__ __forceinline__ void init(const dec_args & a, const int32_t * table, int32_t split, int64_t b, int64_t e,
                                         int32_t lane, int64_t ctx) {
        if (a.strided) {
            const int32_t s = seq_of(a, split);
            const int32_t j = split - a.split0[s], n = a.split0[s + 1] - a.split0[s];
            const int32_t tiles_cap = static_cast<int32_t>((a.ctx[s] + kTileTokens - 1) / kTileTokens);
            const int32_t cap_n = tiles_cap > j ? (tiles_cap - j + n - 1) / n : 0;
            page_lane = page_of(table, lane < cap_n, (j + n * lane) >> 3);
            page_hi = page_of(table, 64 + lane < cap_n, (j + n * (64 + lane)) >> 3);
            g0 = j;
            stride = n;
            recount(ctx);
        } else {
            g0 = static_cast<int32_t>(b / kTileTokens);
            stride = 1;
            n_tiles = static_cast<int32_t>((e - b + kTileTokens - 1) / kTileTokens);
            page_lane = page_of(table, lane < n_tiles, (g0 + lane) >> 3);
            page_hi = page_of(table, 64 + lane < n_tiles, (g0 + 64 + lane) >> 3);
        }
    }
    // A strided walk sized by the host's bound: its tile count for the sequence's actual context (read from the
    // device after the page lookups were issued)
    __device__ __forceinline__ void recount(int64_t ctx) {
        const int32_t tiles = static_cast<int32_t>((ctx + kTileTokens - 1) / kTileTokens);
        n_tiles = tiles > g0 ? (tiles - g0 + stride - 1) / stride : 0;
    }
    // A walk tile whose page is not mapped (page-table entry -1: the slot was trimmed under a captured launch, outside
    // the contract): its lanes read page 0 instead, so nothing faults, and the workgroup is told (uniform) so that it
    // writes no output for its sequence (its partials carry a NaN max: the merge writes nothing for such a row).
    // Lanes past the walk take page 0 too. Every dense walk calls this once its tile count is final.
    __device__ __forceinline__ bool guard_unmapped(int32_t lane) {
        const bool neg = lane < n_tiles && page_lane < 0, neg_hi = 64 + lane < n_tiles && page_hi < 0;
        if (neg || lane >= n_tiles) {
            page_lane = 0;
        }
        if (neg_hi || 64 + lane >= n_tiles) {
            page_hi = 0;
        }
        return __any(neg || neg_hi);
    }
    // byte offset of walk tile ti within the (layer, head) plane of the pool
    __device__ __forceinline__ int64_t tile_off(const pool_view & pv, int32_t ti) const {
        const int32_t lo = __builtin_amdgcn_readlane(page_lane, ti & 63);
        const int32_t hi = __builtin_amdgcn_readlane(page_hi, ti & 63);
        const int32_t phys = ti < 64 ? lo : hi;
        return int64_t(phys) * pv.page_stride + int64_t((g0 + stride * ti) & 7) * kTileBytes;
    }
    // the first cell of walk tile ti
    __device__ __forceinline__ int64_t tok0(int32_t ti) const { return int64_t(g0 + stride * ti) * kTileTokens; }
};

// A sequence's context: the host's, or the device word's (ctx_dev)
__device__ __forceinline__ int64_t seq_ctx(const dec_args & a, int32_t s) {
    if (a.ctx_dev != nullptr) {
        // a vector load: a scalar one would hold up every later kernel-argument read until it returned
        return *(const volatile __attribute__((address_space(1))) int64_t *)(a.ctx_dev + s);
    }
    return a.ctx[s];
}

// A device context outside T .. the host's bound: the sequence's workgroups write nothing (its first workgroup sets
// the error bit). Uniform across the workgroup.
__device__ __forceinline__ bool refused(const dec_args & a, int32_t s, int64_t ctx, int32_t sp, int32_t kvh) {
    if (a.ctx_dev != nullptr && (ctx < a.T || ctx > a.ctx[s])) {
        if (sp == 0 && kvh == 0 && threadIdx.x == 0 && a.err != nullptr) {
            atomicOr(a.err, FNKV_DEV_ERR_DEPTH);
        }
        return true;
    }
    return false;
}

// A dense walk over an unmapped page (split_src::guard_unmapped): with a device word, FNKV_DEV_ERR_DEPTH is set
__device__ __forceinline__ void report_unmapped(const dec_args & a, bool unmapped) {
    if (unmapped && threadIdx.x == 0 && a.err != nullptr) {
        atomicOr(a.err, FNKV_DEV_ERR_DEPTH);
    }
}

// the step token of this lane's query row (rt * 16 + j); padding rows take the last
__device__ __forceinline__ int32_t t_of_row(const dec_args & a, int32_t rt, int32_t j) {
    const int32_t row = rt * 16 + j;
    return row < a.R ? row / a.G : a.T - 1;
}

// An attention launch's outputs (finish4, gather.h): plain fp16 [rows][hq][256] in `out`, or with `gate` set (row r's
// gates at gate + r gate_stride) the gated F32 value in out_f32 and its int8 activation format (codes [rows][256],
// act_scales [rows][8][2]); with out16 set instead (prompt rows, out_f32 optional) the gated fp16 value, bit 0 of *err
// set for a value that fp16 cannot hold (|x| > 65,504, or NaN)
struct out_args {
    uint16_t * out = nullptr;
    const float * gate = nullptr;
    int32_t gate_stride = 0;
    float * out_f32 = nullptr;
    int8_t * codes = nullptr;
    float * act_scales = nullptr;
    uint16_t * out16 = nullptr;
    uint32_t * err = nullptr;
};

// the split merge's arguments: partials of n_seq sequences (the rows of a sparse launch are sequences of one token)
struct merge_args {
    const float * po;
    const float * pml;
    out_args fin;
    int32_t T, G, hq, R, h_kv, n_seq;
    int32_t split0[FNKV_MAX_SEQS + 1]; // dense: sequence s's splits are split0[s] .. split0[s + 1] - 1
    // sparse: every row holds sel_splits splits, row s (position depth + s) partials in the first of them that its
    // selection's tiles reach; 0: dense
    int32_t sel_splits = 0;
    int64_t depth = 0;
    // the launch's device word (dec_args, gather_args): a refused sequence's (or sparse launch's) outputs are left as
    // they were; dense strided splits past a shorter context hold nothing
    const int64_t * ctx_dev = nullptr;
    const int32_t * depth_dev = nullptr;
    int64_t cap[FNKV_MAX_SEQS] = {0};
    int32_t T_dev = 0; // the launch's step tokens (rows of a sparse launch)
};

class kv_pool;
struct fused_prep; // gather.h
// host: the merge launch (decode.hip)
void launch_merge(const merge_args & m, hipStream_t st);
// host: the dense launch's one-stream-a-wave kernel for NT = 1 .. 3 row tiles (stream.hip)
void launch_stream(int32_t device, int32_t NT, dim3 grid, const dec_args & a, hipStream_t st);
// the split size (cells) of a dense launch run by the stream kernel with NT row tiles; fine: kFineSplit is allowed;
// max_splits: at most this many splits
constexpr int32_t kFineSplit = 128;
constexpr int64_t kAnySplits = int64_t(1) << 40;
struct split_choice {
    int32_t cells = 0; // a split's
    // the best split of at most 64 tiles: the workspace asked for holds its partials too, so the size asked for is no
    // smaller where a launch takes longer splits (fewer partials)
    int32_t asked = 0;
};
split_choice choose_split_stream(int32_t n_seq, const int64_t * ctx, int32_t h_kv, int32_t cus, int32_t NT, bool fine,
                                 int64_t max_splits = kAnySplits);
// a launch's depth read from device memory (the reference's depth word, attend.h:108): depth + T <= max_cells or
// the launch writes nothing and ORs FNKV_DEV_ERR_DEPTH into *err
struct dev_depth {
    const int32_t * depth;
    int64_t max_cells;
    uint32_t * err;
};
// host: a sparse launch of decode rows over the pool (sparse.hip), with gated outputs when `gate` is set.
// dd set: `depth` is not read; the plan (grid, workspace) follows from dd->max_cells. q_lo set: q's fp16 low parts
// beside q (gather_args::q_lo), 16-byte aligned
int sparse_launch(const fnkv_pool * pool, int32_t slot, int64_t depth, int32_t T, int32_t layer, int32_t hq, float scale,
                  const void * q, const void * body, const void * offsets, const void * k_new, const void * v_new,
                  int32_t new_dtype, void * out, const out_args * gate, void * ws, int64_t ws_bytes,
                  hipStream_t st, const char * who, const fused_prep * fp = nullptr, const dev_depth * dd = nullptr,
                  const uint16_t * q_lo = nullptr);
// host: the sparse launch of `rows` prompt rows at positions pos0 .. (qsp.hip checks the call; sparse.hip): the
// workspace its splits' partials need, and the launch with the gated outputs
int64_t prompt_ws_bytes(const kv_pool & p, int64_t pos0, int32_t rows, int32_t G);
int prompt_launch(const kv_pool & p, int32_t slot, int32_t layer, int32_t pos0, int32_t rows, int32_t hq,
                  const uint32_t * body, const int32_t * offsets, const fused_prep & fp, const out_args & fin, void * ws,
                  hipStream_t st);

__device__ __forceinline__ int32_t seq_of(const dec_args & a, int32_t split) {
    int32_t s = 0;
    while (s + 1 < a.n_seq && a.split0[s + 1] <= split) {
        ++s;
    }
    return s;
}

// The step's new cells ctx - T .. ctx - 1 that fall in this split [begin, end): quantized and written here (each
// position lies in exactly one split, so one workgroup writes it and only that workgroup reads it in this launch).
// The barrier's workgroup-scope release / acquire makes the stores visible to the workgroup's own later loads; an
// agent-scope fence would write back and invalidate the whole L2 under every other workgroup's stream.
template <int WAVES>
__device__ __forceinline__ void append_new_cells(const dec_args & a, const int32_t * table, int32_t s, int32_t kvh,
                                                 int64_t ctx, int64_t begin, int64_t end, int32_t sj, int32_t sn,
                                                 int32_t wave, int32_t lane) {
    if (a.k_new == nullptr) {
        return;
    }
    const pool_view & pv = a.pv;
    const int64_t first_new = ctx - a.T;
    // a new cell is written by the workgroup whose walk holds its tile: the split of its cell range, or (strided,
    // sn splits) split tile % sn
    for (int32_t job = wave; job < 2 * a.T; job += WAVES) {
        const int64_t pos = first_new + (job >> 1);
        const bool mine = sn != 0 ? static_cast<uint32_t>(pos >> 5) % static_cast<uint32_t>(sn) == static_cast<uint32_t>(sj)
                                  : (pos >= begin && pos < end);
        if (!mine) {
            continue;
        }
        const int32_t kv = job & 1;
        if (table[pos >> 8] < 0) {
            continue; // an unmapped page (outside the contract): nothing is written
        }
        const int64_t src = ((int64_t(s) * a.T + (pos - first_new)) * pv.h_kv + kvh) * kHeadDim;
        float x[4];
        if (a.new_f32) {
            load4<true>(static_cast<const float *>(kv ? a.v_new : a.k_new) + src, lane, x);
        } else {
            load4<false>(static_cast<const uint16_t *>(kv ? a.v_new : a.k_new) + src, lane, x);
        }
        quantize_store_fmt(x, lane, tile_of(pv, table, a.layer, kvh, pos), static_cast<int32_t>(pos & 31), kv,
                           pv.format);
    }
    __syncthreads();
}

// The scores' optional second Q operand: none (q is the fp16 operand alone), or q's fp16 low parts, block b's from
// qlo(b), chained into the same MFMA results as the hi parts (the K codes then enter exactly, without the bias).
struct no_qlo {
    __device__ half8 operator()(int) const { return half8{}; }
};
template <typename QLOP> constexpr bool has_qlo = !std::is_same<QLOP, no_qlo>::value;

// sig: the row's per-block sums of q (the bias correction's operand), as fp16 hi (qg = 0) and lo (qg = 1) parts. The
// sums are products with a row of ones (every lane of row j gets its block's sum): 8 MFMAs and 50 VALU instructions in
// place of about 210, which every wave of a launch runs before its first tile.
__device__ __forceinline__ half8 q_sums(const half8 (&qop)[kBlocks], int32_t qg) {
    const _Float16 one = static_cast<_Float16>(1.0f);
    const half8 ones8 = {one, one, one, one, one, one, one, one};
    half8 sig;
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
        const float sigma = mfma16(ones8, qop[b], floatx4{0.0f, 0.0f, 0.0f, 0.0f})[0];
        const _Float16 hi = static_cast<_Float16>(sigma);
        const _Float16 lo = static_cast<_Float16>(sigma - static_cast<float>(hi));
        sig[b] = qg == 0 ? hi : qg == 1 ? lo : static_cast<_Float16>(0.0f);
    }
    return sig;
}

// The lazily moved softmax reference: a row's running max moves only when a tile's max exceeds it by more than this many
// log2 units, so the rescale of the accumulators is rare and a weight times a V scale (at most 65504 / 127) stays
// inside fp16
constexpr float kLazyLog2 = 6.0f;

} // namespace fnkv
