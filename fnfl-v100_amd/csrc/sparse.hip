// Sparse (QSA) attention at decode rows: each of T <= 5 query rows of one sequence attends only to its selection —
// the reference's selected-block body (fn/kernels/qsa/qsa.h:77-81: per row K ascending 4-cell block IDs, then its
// tail cells), at most 512 blocks and 3 tail cells a row — instead of its whole causal context. This is the reference's
// production decode path (attn::attend over the body, fn/kernels/qsa/attend.h:97-141, cell expansion
// attend.cu:405-421), here over the Q8_0 / KV8 pool.
//
// The kernel is gather.hip's (eight selected blocks a virtual tile, each lane loading its own block's bytes); here are
// the launches' checks and plans. A row's new cell is written by the workgroups that read its block (several rows
// without a prepare: by an append launch first, since a row may read an earlier row's cell); the rows of one launch run
// side by side, each as its own splits, and merge_kernel folds the splits that held some of a row's tiles.
#include "../../include/fnkv.h"
#include "common.h"
#include "layout.h"
#include "mfma.h"
#include "q8_0.h"
#include "decode_common.h"
#include "gather.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

namespace fnkv {

// The launch shape of `rows` rows, the deepest at position last: each row's splits, whether a wave takes several tiles,
// and the partials of every split (a row of one split writes none, its region is unused).
//   * Decode rows (at most kSelMaxRows): one virtual tile a wave, the row's at most 65 tiles over at most 17 splits. A
//     step has few rows, so its time is one tile's latency, and fewer, longer splits leave the device idle. That form
//     holds one workgroup a CU; (row, head tile) pairs whose splits are more than the CUs (from 16 on) take the splits
//     that one round holds, several tiles a wave: attn::attend of 5 rows of 32 heads on 8 KV heads at 3,000 cells 37.7 ->
//     26.4 us a layer (a kernel that read whole tiles: 28.8), at 100,000 41.3 -> 29.4; without prepare and gate 33.4 ->
//     24.6 (25.9); two rounds of workgroups a CU where they fit: 26.3.
//   * Prompt rows: the splits that bring the launch to at most two workgroups a CU (what its LDS lets run at once): one
//     where the (row, head tile) pairs are more than the CUs. Such rows need no partials and no merge.
struct sparse_plan {
    int32_t n_splits = 0;
    bool many = false;
    int64_t pml_off = 0, bytes = 0;
};
sparse_plan plan_sparse(const kv_pool & p, int64_t last, int32_t rows, int32_t G) {
    sparse_plan pl;
    // the deepest row's blocks and one tail entry (which rows have a tail follows from each row's own position)
    const int32_t entries = sel_shape(static_cast<int32_t>(std::min<int64_t>(last, kSelMaxCells))).K + 1;
    const int32_t full = (entries + 8 * kGatherWaves - 1) / (8 * kGatherWaves);
    pl.n_splits = full;
    const int64_t cus = device_cus(p.device()), pairs = int64_t(rows) * p.h_kv() * ((G + 15) / 16);
    const bool over = rows <= kSelMaxRows && pairs * full > cus;
    if (rows > kSelMaxRows || over) {
        pl.n_splits =
            static_cast<int32_t>(std::min<int64_t>(full, std::max<int64_t>(1, (over ? 1 : 2) * cus / pairs)));
    }
    pl.many = pl.n_splits < full || over;
    auto up16 = [](int64_t x) { return (x + 15) & ~int64_t(15); };
    const int64_t head_rows = int64_t(p.h_kv()) * G;
    pl.pml_off = rows * pl.n_splits * head_rows * kHeadDim * 4;
    // what the workspace is asked to hold: no fewer row splits than any smaller launch writes, so that one sized for a
    // caller's largest chunk serves its smaller ones (which take more splits a row); rows of one split write none
    const int64_t fill = std::max<int64_t>(2 * cus / (int64_t(p.h_kv()) * ((G + 15) / 16)),
                                           int64_t(kSelMaxRows) * full);
    const int64_t units = std::min<int64_t>(int64_t(rows) * full, fill);
    pl.bytes = up16(units * head_rows * (kHeadDim + 2) * 4);
    return pl;
}

// the kernel, then the merge when a row has several splits
int sparse_enqueue(const kv_pool & p, int32_t slot, const sparse_plan & pl, gather_args & a, void * ws, hipStream_t st) {
    a.pv = p.view();
    a.table = a.pv.table + int64_t(slot) * a.pv.table_stride;
    a.n_splits = pl.n_splits;
    a.many = pl.many ? 1 : 0;
    a.head_tiles = (a.G + 15) / 16;
    a.po = static_cast<float *>(ws);
    a.pml = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + pl.pml_off);
    launch_gather(p.device(), a, st);
    if (pl.n_splits > 1) {
        merge_args m;
        m.po = a.po;
        m.pml = a.pml;
        m.fin = a.fin;
        m.T = 1; // the rows fold as sequences of one step token each
        m.G = a.G;
        m.hq = a.hq;
        m.R = a.G;
        m.h_kv = p.h_kv();
        m.n_seq = a.T;
        m.sel_splits = pl.n_splits;
        m.depth = a.depth;
        m.depth_dev = a.depth_dev;
        m.cap[0] = a.cap;
        m.T_dev = a.T;
        launch_merge(m, st);
    }
    return hipGetLastError() == hipSuccess ? FNKV_OK : FNKV_ERR_HIP;
}

// The sparse launch of decode rows; `gate` set: the gated F32 output and its activation format instead of the fp16
// out. Returns a status; nothing is enqueued unless it is FNKV_OK.
int sparse_launch(const fnkv_pool * pool, int32_t slot, int64_t depth, int32_t T, int32_t layer, int32_t hq, float scale,
                  const void * q, const void * body, const void * offsets, const void * k_new, const void * v_new,
                  int32_t new_dtype, void * out, const out_args * gate, void * ws, int64_t ws_bytes,
                  hipStream_t st, const char * who, const fused_prep * fp, const dev_depth * dd,
                  const uint16_t * q_lo) {
    const kv_pool * p = pool_of(pool);
    const std::string name(who);
    if (dd != nullptr) { // the plan is the bound's: the deepest rows' tiles
        if (dd->depth == nullptr || dd->err == nullptr || (reinterpret_cast<uintptr_t>(dd->depth) & 3) != 0 ||
            (reinterpret_cast<uintptr_t>(dd->err) & 3) != 0 || dd->max_cells < T) {
            set_error(name + ": the device depth and error words (4-byte aligned) and max_cells >= rows required");
            return FNKV_ERR_ARG;
        }
        depth = dd->max_cells - T;
    }
    if (p == nullptr || slot < 0 || slot >= p->pages().n_slots() || T <= 0 || T > kSelMaxRows || depth < 0 ||
        layer < 0 || layer >= p->layers() || hq <= 0 || hq % p->h_kv() != 0 || q == nullptr || body == nullptr ||
        offsets == nullptr || (out == nullptr && gate == nullptr) || ws == nullptr || !(scale > 0.0f) ||
        !std::isfinite(scale) || ((k_new == nullptr) != (v_new == nullptr)) ||
        (new_dtype != FNKV_F16 && new_dtype != FNKV_F32)) {
        set_error(name + ": argument outside the contract");
        return FNKV_ERR_ARG;
    }
    const int32_t G = hq / p->h_kv();
    const int64_t ctx = depth + T;
    if (G > FNKV_MAX_ROWS || ctx > kSelMaxCells || ctx > p->mapped_cells(slot)) {
        set_error(name + ": G = " + std::to_string(G) + " (at most " + std::to_string(FNKV_MAX_ROWS) +
                  ") or cells " + std::to_string(ctx) + " outside the slot's mapped cells (at most " +
                  std::to_string(kSelMaxCells) + ")");
        return FNKV_ERR_ARG;
    }
    if ((reinterpret_cast<uintptr_t>(q) & 15) != 0 || (reinterpret_cast<uintptr_t>(q_lo) & 15) != 0 || (reinterpret_cast<uintptr_t>(out) & 15) != 0 ||
        (reinterpret_cast<uintptr_t>(ws) & 15) != 0 || (reinterpret_cast<uintptr_t>(body) & 3) != 0 ||
        (reinterpret_cast<uintptr_t>(offsets) & 3) != 0) {
        set_error(name + ": q, out and ws must be 16-byte aligned, body and offsets 4-byte aligned");
        return FNKV_ERR_ARG;
    }
    const sparse_plan pl = plan_sparse(*p, ctx - 1, T, G);
    if (ws_bytes < pl.bytes) {
        set_error(name + ": workspace too small");
        return FNKV_ERR_ARG;
    }
    // several rows: their new cells first (a row may read an earlier row's new cell; the rows run side by side); one
    // row of one tile a wave: the launch writes it, by the split that reads its tile
    if (fp != nullptr && (G > 16 || fp->rows != T)) {
        set_error(name + ": a launch that prepares its rows takes at most 16 query heads a KV head");
        return FNKV_ERR_ARG;
    }
    if (k_new != nullptr && (T > 1 || pl.many) && fp == nullptr) {
        if (append_enqueue(*p, slot, layer, depth, dd != nullptr ? dd->depth : nullptr, ctx, T, k_new, v_new,
                           new_dtype, st) != FNKV_OK) {
            set_error(name + ": launch failed");
            return FNKV_ERR_HIP;
        }
    }
    gather_args a = {};
    a.layer = layer;
    a.T = T;
    a.G = G;
    a.hq = hq;
    a.depth = depth;
    a.cap = ctx;
    if (dd != nullptr) {
        a.depth_dev = dd->depth;
        a.err = dd->err;
    }
    a.body = static_cast<const uint32_t *>(body);
    a.q = static_cast<const uint16_t *>(q);
    a.q_lo = q_lo;
    if (fp != nullptr) {
        a.fp = *fp;
    } else if (T == 1 && !pl.many) {
        a.k_new = k_new;
        a.v_new = v_new;
        a.new_f32 = new_dtype == FNKV_F32 ? 1 : 0;
    }
    a.c2 = scale * 1.4426950408889634f;
    if (gate != nullptr) {
        a.fin = *gate;
    } else {
        a.fin.out = static_cast<uint16_t *>(out);
    }
    if (sparse_enqueue(*p, slot, pl, a, ws, st) != FNKV_OK) {
        set_error(name + ": launch failed");
        return FNKV_ERR_HIP;
    }
    return FNKV_OK;
}

// Prompt rows (qsp_attend): each over its own selection body (the slab layout), its query heads formed by the launch.
// The caller has checked the arguments; ws holds prompt_ws_bytes.
int64_t prompt_ws_bytes(const kv_pool & p, int64_t pos0, int32_t rows, int32_t G) {
    return plan_sparse(p, pos0 + rows - 1, rows, G).bytes;
}

int prompt_launch(const kv_pool & p, int32_t slot, int32_t layer, int32_t pos0, int32_t rows, int32_t hq,
                  const uint32_t * body, const int32_t * offsets, const fused_prep & fp, const out_args & fin, void * ws,
                  hipStream_t st) {
    gather_args a = {};
    a.layer = layer;
    a.T = rows;
    a.G = hq / p.h_kv();
    a.hq = hq;
    a.depth = pos0;
    a.body = body;
    a.offsets = offsets;
    a.fp = fp;
    a.c2 = (1.0f / 16.0f) * 1.4426950408889634f;
    a.fin = fin;
    return sparse_enqueue(p, slot, plan_sparse(p, int64_t(pos0) + rows - 1, rows, a.G), a, ws, st);
}

} // namespace fnkv

using fnkv::set_error;

extern "C" {

int64_t fnkv_sparse_workspace_bytes(const fnkv_pool * pool, int64_t depth, int32_t T, int32_t hq) {
    const fnkv::kv_pool * p = fnkv::pool_of(pool);
    if (p == nullptr || T <= 0 || T > fnkv::kSelMaxRows || depth < 0 || hq <= 0 || hq % p->h_kv() != 0) {
        return -1;
    }
    return fnkv::plan_sparse(*p, depth + T - 1, T, hq / p->h_kv()).bytes;
}

int fnkv_attn_sparse(const fnkv_pool * pool, int32_t slot, int64_t depth, int32_t T, int32_t layer, int32_t hq,
                     float scale, const void * q, const void * body, const void * offsets, const void * k_new,
                     const void * v_new, int32_t new_dtype, void * out, void * ws, int64_t ws_bytes, void * stream) {
    return fnkv::sparse_launch(pool, slot, depth, T, layer, hq, scale, q, body, offsets, k_new, v_new,
                               new_dtype, out, nullptr, ws, ws_bytes, static_cast<hipStream_t>(stream),
                               "fnkv_attn_sparse");
}

int fnkv_attn_sparse_dev(const fnkv_pool * pool, int32_t slot, const int32_t * depth, int64_t max_cells, int32_t T,
                         int32_t layer, int32_t hq, float scale, const void * q, const void * body,
                         const void * offsets, const void * k_new, const void * v_new, int32_t new_dtype, void * out,
                         void * ws, int64_t ws_bytes, uint32_t * err, void * stream) {
    const fnkv::dev_depth dd = {depth, max_cells, err};
    return fnkv::sparse_launch(pool, slot, 0, T, layer, hq, scale, q, body, offsets, k_new, v_new, new_dtype, out,
                               nullptr, ws, ws_bytes, static_cast<hipStream_t>(stream), "fnkv_attn_sparse_dev",
                               nullptr, &dd);
}

} // extern "C"
