// The sparse attention launch (gather.hip): its arguments, a row's selection, and the output forms it shares with the
// split merge (decode.hip).
#pragma once

#include "decode_common.h"
#include "layout.h"
#include "mfma.h"
#include "rope.h"

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>

namespace fnkv {

constexpr int32_t kSelMaxCells = 262144 + 32; // the reference's max_cells
constexpr int32_t kSelTopBlocks = 512;        // blocks a row (qsa.h)
constexpr int32_t kSelMaxRows = 5;            // decode rows a launch
constexpr int32_t kSlabRows = 128;            // prompt rows a slab (qsa_prompt.h prompt_slab)
constexpr int64_t kSlabWords = int64_t(kSlabRows) * (2 + kSelTopBlocks + 3); // a slab's bodies (max_row_words each)
constexpr int32_t kGatherWaves = 4;           // waves a workgroup

// The selection of the row at position q (fn/kernels/qsa/qsa.h:77-81): K 4-cell blocks of the n_vis whole ones, then
// `tail` cells of block n_vis; entries 8 t .. 8 t + 7 (the tail is entry K) are virtual tile t
struct sel_shape {
    int32_t n_vis, K, tail, tiles;
    __host__ __device__ explicit sel_shape(int32_t q)
        : n_vis((q + 1) / 4), K(n_vis < kSelTopBlocks ? n_vis : kSelTopBlocks), tail((q + 1) % 4),
          tiles((K + (tail != 0 ? 1 : 0) + 7) / 8) {}
};

// Inputs of a launch that prepares its rows: each workgroup forms its query heads (F32 RMS norm and IMROPE) while its
// blocks load, and the ones that read a new cell write the cell's K (normed, roped) and V in the pool's format first.
struct fused_prep {
    const float * qfull = nullptr; // [rows][hq][512]: each head's q, then its gate; null: the launch reads q
    const float * kv_k = nullptr;  // [rows][h_kv][256], or null: the rows' cells are written already
    const float * kv_v = nullptr;  // [rows][h_kv][256]
    const float * q_norm = nullptr;
    const float * k_norm = nullptr;
    const int32_t * pos = nullptr; // [4][rows] (row_major: [rows][4]); null: row z at pos0 + z on every plane
    int32_t row_major = 0;
    int32_t pos0 = 0;
    float theta_scale = 0.0f;
    float * q_f32 = nullptr; // optional [rows][hq][256]
    float * k_f32 = nullptr; // optional [rows][h_kv][256]
    int32_t rows = 1;        // the call's rows
};

struct gather_args {
    pool_view pv;
    const int32_t * table; // the slot's page table
    int32_t layer, T, G, hq, n_splits;
    int32_t head_tiles;          // 16-head tiles a KV head
    int32_t many;                // a wave may take several virtual tiles
    int64_t depth;               // row z is at position depth + z
    const int32_t * depth_dev;   // set: the depth is this device word, and depth + T <= cap or nothing is written
    int64_t cap;
    uint32_t * err;
    const uint32_t * body;       // the rows' selection bodies, packed in order (qsa.h:77-81), or
    const int32_t * offsets;     // set: in slabs of kSlabRows rows, row r's at byte offsets[129 (r / 128) + r % 128]
    const uint16_t * q;          // fp16 [T][hq][256]; unused by a launch that prepares its rows
    const uint16_t * q_lo;       // set: q's fp16 low parts (a launch that prepares its rows reads only its presence)
    const void * k_new;          // one row's new cell [h_kv][256], or null
    const void * v_new;
    int32_t new_f32;
    fused_prep fp;
    float c2;                    // scale * log2(e)
    float * po;                  // [T][n_splits][h_kv][G][256] partial accumulators (n_splits > 1)
    float * pml;                 // ... their (m, l)
    out_args fin;                // the outputs of rows with one split
};

void launch_gather(int32_t device, const gather_args & a, hipStream_t st);

// Online softmax (base 2) of a virtual tile's scores for this lane's row: its cells r < n0 of the first half and
// r < n1 of the second are attended. The row's reference m_run moves only when the tile's max exceeds it by more than
// kLazyLog2 (alpha: the factor its accumulators take before this tile's terms), so a weight stays <= 2^kLazyLog2 and
// a weight times a V scale inside fp16. EXACT_MAX (q as hi + lo): m_run follows every new max and the weights carry
// 2^kLazyLog2, which cancels in every fold; a weight times a V scale then keeps 6 more bits above fp16's subnormals.
template <bool EXACT_MAX>
__device__ __forceinline__ void gather_softmax(const floatx4 (&sc)[2], int32_t n0, int32_t n1, float c2, float & m_run,
                                               float & l_run, float (&pf)[8], float & alpha) {
    float raw[8];
    float mx = kNegInf;
    if (__all(n0 == 4 && n1 == 4)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            raw[i] = sc[i >> 2][i & 3];
            mx = fmaxf(mx, raw[i]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            raw[i] = (i & 3) < (i < 4 ? n0 : n1) ? sc[i >> 2][i & 3] : kNegInf;
            mx = fmaxf(mx, raw[i]);
        }
    }
    mx = rows_max(mx) * c2;
    const bool move = mx > m_run + (EXACT_MAX ? 0.0f : kLazyLog2); // m_run = -inf: any visible score moves it
    const float m_new = move ? mx : m_run;
    const float m_use = m_new == kNegInf ? 0.0f : m_new;
    alpha = move ? __builtin_amdgcn_exp2f(m_run - m_use) : 1.0f;
    const float m_pf = EXACT_MAX ? m_use - kLazyLog2 : m_use;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        pf[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(raw[i], c2, -m_pf));
    }
    l_run = __builtin_fmaf(l_run, alpha, sum8(pf));
    m_run = m_new;
}

// Four values c0 .. c0 + 3 of an output row (row = token * hq + head) from their folded accumulators A and the row's
// L: A / L as fp16.
__device__ __forceinline__ void finish_plain(const out_args & o, int64_t row, int32_t c0, floatx4 A, float L) {
    const float inv = 1.0f / L;
    uint2 pk;
    pk.x = uint32_t(__half_as_ushort(__float2half_rn(A[0] * inv))) |
           (uint32_t(__half_as_ushort(__float2half_rn(A[1] * inv))) << 16);
    pk.y = uint32_t(__half_as_ushort(__float2half_rn(A[2] * inv))) |
           (uint32_t(__half_as_ushort(__float2half_rn(A[3] * inv))) << 16);
    *reinterpret_cast<uint2 *>(o.out + row * kHeadDim + c0) = pk;
}
// The gated form (fn/kernels/qsa/attend.cu:619-655's finish): A / L / (1 + exp(-gate)) in F32, with the prompt path's
// fp16 output or the int8 activation format of the 32-value run, whose 8 lanes are consecutive and all take part. g4: the
// four gates (finish_gate), for callers that request them early.
__device__ __forceinline__ float4 finish_gate(const out_args & o, int64_t row, int32_t c0) {
    return *reinterpret_cast<const float4 *>(o.gate + row * o.gate_stride + c0);
}
__device__ __forceinline__ void finish_gated(const out_args & o, int64_t row, int32_t c0, floatx4 A, float L, float4 g4) {
    const float gr[4] = {g4.x, g4.y, g4.z, g4.w};
    float y[4];
#pragma unroll
    for (int32_t e = 0; e < 4; ++e) {
        y[e] = A[e] / L * (1.0f / (1.0f + expf(-gr[e])));
    }
    if (o.out_f32 != nullptr) {
        *reinterpret_cast<float4 *>(o.out_f32 + row * kHeadDim + c0) = make_float4(y[0], y[1], y[2], y[3]);
    }
    if (o.out16 != nullptr) {
        bool bad = false;
        uint16_t hb[4];
#pragma unroll
        for (int32_t e = 0; e < 4; ++e) {
            bad = bad || !(fabsf(y[e]) <= 65504.0f);
            hb[e] = __half_as_ushort(__float2half_rn(y[e]));
        }
        *reinterpret_cast<uint2 *>(o.out16 + row * kHeadDim + c0) =
            make_uint2(uint32_t(hb[0]) | (uint32_t(hb[1]) << 16), uint32_t(hb[2]) | (uint32_t(hb[3]) << 16));
        if (bad && o.err != nullptr) {
            atomicOr(o.err, 1u);
        }
        return;
    }
    int8_t q[4];
    float ds[2];
    act_run<4, 8>(y, q, ds);
    *reinterpret_cast<uint32_t *>(o.codes + row * kHeadDim + c0) =
        uint32_t(uint8_t(q[0])) | (uint32_t(uint8_t(q[1])) << 8) | (uint32_t(uint8_t(q[2])) << 16) |
        (uint32_t(uint8_t(q[3])) << 24);
    if ((c0 & 31) == 0) {
        *reinterpret_cast<float2 *>(o.act_scales + (row * 8 + c0 / 32) * 2) = float2{ds[0], ds[1]};
    }
}
// either, by the launch's outputs
__device__ __forceinline__ void finish4(const out_args & o, int64_t row, int32_t c0, floatx4 A, float L, float4 g4) {
    if (o.gate == nullptr) {
        finish_plain(o, row, c0, A, L);
    } else {
        finish_gated(o, row, c0, A, L, g4);
    }
}

} // namespace fnkv
