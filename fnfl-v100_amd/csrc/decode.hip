// Decode and speculative-verify attention over the Q8_0 page pool (T = 1 .. 6 query tokens a sequence), split-K
// over pages with a log-sum-exp merge: the dense launches' host side (fnkv_attn_decode, _dev, _noalloc; their kernel
// is stream.hip's) and the split merge of the dense and the sparse launches (gather.hip).
//
// What the launches compute (the reference's decode attention, fn/kernels/qsa/attend.h:8-34; dense: causal over the
// whole context, on the pool's 8-bit format): for query row (t, head h) of a sequence holding ctx cells,
//   o = sum_c softmax_c(q . k_c * scale) v_c over cells c <= ctx - T + t (sparse: over the row's selected cells),
// with k_c, v_c the decoded values (code * fp32(d)); scores, softmax statistics and accumulators in fp32; fp16
// out. The split-K partials (m, l, acc) fold in a fixed order as the reference's finish does (attend.cu:621-655):
// M = max m_j, L = sum l_j e^(m_j - M), A = sum acc_j e^(m_j - M), o = A / L.
#include "../../include/fnkv.h"
#include "common.h"
#include "layout.h"
#include "mfma.h"
#include "q8_0.h"
#include "decode_common.h"
#include "gather.h"

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

namespace fnkv {

// The splits of sequence s that hold partials: its first s0 and count n; false when the launch refused the sequence
// (its outputs are left as they were). SPARSE: the rows of a sparse launch (merge_args::sel_splits).
template <bool SPARSE>
__device__ __forceinline__ bool merge_splits(const merge_args & a, int32_t s, int32_t & s0, int32_t & n) {
    if constexpr (SPARSE) { // row s's splits that held some of its virtual tiles
        int64_t d = a.depth;
        if (a.depth_dev != nullptr) {
            d = *a.depth_dev;
            if (d < 0 || d + a.T_dev > a.cap[0]) {
                return false;
            }
        }
        const int32_t used = (sel_shape(static_cast<int32_t>(d) + s).tiles + kGatherWaves - 1) / kGatherWaves;
        s0 = s * a.sel_splits;
        n = used < a.sel_splits ? used : a.sel_splits;
        return true;
    }
    s0 = a.split0[s];
    n = a.split0[s + 1] - s0;
    if (a.ctx_dev != nullptr) { // a device context: strided splits past its tiles held nothing
        const int64_t c = a.ctx_dev[s];
        if (c < a.T_dev || c > a.cap[s]) {
            return false;
        }
        const int64_t tiles = (c + kTileTokens - 1) / kTileTokens;
        n = tiles < n ? static_cast<int32_t>(tiles) : n;
    }
    return true;
}

// Fold the splits of each (sequence, KV head, row) of a dense launch with more than kRowMergeSplits splits a sequence:
// one workgroup a (row, 32 values); 256 threads = 8 float4 columns x 32 split groups. Group g folds splits g, g + 32, ...
// in order with a running max (all its loads independent, so they are in flight together: one memory round trip), then
// the 32 groups fold in order in LDS (deterministic: the same order for every launch).
__global__ __launch_bounds__(256) void merge_kernel(merge_args a) {
    __shared__ float sM[4];
    __shared__ float sL[4];
    __shared__ floatx4 sA[4][8];
    const int32_t tid = static_cast<int32_t>(threadIdx.x);
    const int32_t c4 = tid & 7, g = tid >> 3;
    const int32_t chunk = static_cast<int32_t>(blockIdx.x) & 7;
    int32_t rest = static_cast<int32_t>(blockIdx.x) >> 3;
    const int32_t r = rest % a.R;
    rest /= a.R;
    const int32_t kvh = rest % a.h_kv;
    const int32_t s = rest / a.h_kv;
    int32_t s0 = 0, n = 0;
    if (!merge_splits<false>(a, s, s0, n)) {
        return;
    }
    float m = kNegInf, l = 0.0f;
    int32_t bad = 0; // a split that saw an unmapped page marked its partial with a NaN max: nothing is written
    floatx4 A = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int32_t i = g; i < n; i += 32) {
        const int64_t prow = (int64_t(s0 + i) * a.h_kv + kvh) * a.R + r;
        const float2 ml = *reinterpret_cast<const float2 *>(a.pml + prow * 2);
        bad |= ml.x != ml.x ? 1 : 0;
        const floatx4 o = *reinterpret_cast<const floatx4 *>(a.po + prow * kHeadDim + chunk * 32 + c4 * 4);
        const float m_new = fmaxf(m, ml.x);
        const float m_use = m_new == kNegInf ? 0.0f : m_new;
        const float f_old = __builtin_amdgcn_exp2f(m - m_use);
        const float f_new = __builtin_amdgcn_exp2f(ml.x - m_use);
        A = A * f_old + o * f_new;
        l = __builtin_fmaf(l, f_old, ml.y * f_new);
        m = m_new;
    }
    // the 32 groups fold pairwise: the wave's 8 by lane exchange (lanes l, l ^ 8, l ^ 16, l ^ 32 share c4), then the
    // 4 waves' results in LDS, in wave order
    auto fold = [](float & m0, float & l0, floatx4 & A0, float m1, float l1, floatx4 A1) {
        const float mn = fmaxf(m0, m1);
        const float mu = mn == kNegInf ? 0.0f : mn;
        const float f0 = __builtin_amdgcn_exp2f(m0 - mu), f1 = __builtin_amdgcn_exp2f(m1 - mu);
        A0 = A0 * f0 + A1 * f1;
        l0 = __builtin_fmaf(l0, f0, l1 * f1);
        m0 = mn;
    };
#pragma unroll
    for (int32_t o = 8; o < 64; o <<= 1) {
        floatx4 A1;
#pragma unroll
        for (int32_t e = 0; e < 4; ++e) {
            A1[e] = __shfl_xor(A[e], o, 64);
        }
        fold(m, l, A, __shfl_xor(m, o, 64), __shfl_xor(l, o, 64), A1);
    }
    const int32_t wave = tid >> 6;
    if ((tid & 63) < 8) {
        sA[wave][c4] = A;
        if (c4 == 0) {
            sM[wave] = m;
            sL[wave] = l;
        }
    }
    if (__syncthreads_or(bad)) {
        return;
    }
    if (tid < 8) {
        float Ms = sM[0], Ls = sL[0];
        floatx4 As = sA[0][tid];
#pragma unroll
        for (int32_t w = 1; w < 4; ++w) {
            fold(Ms, Ls, As, sM[w], sL[w], sA[w][tid]);
        }
        const int32_t t = r / a.G, h = kvh * a.G + r % a.G;
        const int64_t row = (int64_t(s) * a.T + t) * a.hq + h;
        finish_plain(a.fin, row, chunk * 32 + tid * 4, As, Ls);
    }
}

// The split-K fold inside the dense launch (stream.hip) is off by default: measured against the merge kernel on one
// box it is slower (cfg1 43.8-44.2 against 42.0-43.0 us a launch, cfg2 58.9 against 55.0-55.6 us). FNKV_DECODE_FOLD=1
// (read once) or fnkv_test_decode_fold turns it on. The bound of its waits (real-time ticks of 10 ns) is 200 us, far
// past any launch's spread of arrivals; tests lower it to drive the given-up-row path from the host.
std::atomic<int32_t> g_fold_mode{-1}; // -1: the environment's choice
std::atomic<int64_t> g_fold_spin{20000};
bool fold_enabled() {
    const int32_t m = g_fold_mode.load(std::memory_order_relaxed);
    if (m >= 0) {
        return m != 0;
    }
    static const int32_t knob = env_int_once("FNKV_DECODE_FOLD", 0);
    return knob != 0;
}
int64_t fold_spin_ticks() { return g_fold_spin.load(std::memory_order_relaxed); }

int32_t env_int_once(const char * name, int32_t dflt) {
    const char * e = std::getenv(name);
    return e != nullptr ? std::atoi(e) : dflt;
}

int32_t device_cus(int32_t device) {
    // threads racing on the first query each store the same count
    static std::atomic<int32_t> cache[64];
    if (device < 0 || device >= 64) {
        return 256;
    }
    int32_t n = cache[device].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n <= 0) {
            (void)hipGetLastError();
            n = 256;
        }
        cache[device].store(n, std::memory_order_relaxed);
    }
    return n;
}

struct dec_plan {
    int32_t split_tokens = 0, total = 0, strided = 0;
    int32_t split0[FNKV_MAX_SEQS + 1] = {0};
    // the workspace: the fold state (first, at a fixed place: its words persist from launch to launch, zero), then
    // the partials
    int64_t fold_bytes = 0, po_bytes = 0;
    int64_t bytes = 0; // what the workspace is asked to hold (split_choice::asked)
    bool fold = false; // the stream kernel folds the splits itself (no merge launch)
};

int64_t fold_region_bytes(const kv_pool & p) {
    return (int64_t(FNKV_MAX_SEQS) * p.h_kv() * kFoldWords * 4 + 255) & ~int64_t(255);
}
// one split's partials (every KV head's R rows)
int64_t split_bytes(const kv_pool & p, int32_t R) { return int64_t(p.h_kv()) * R * (kHeadDim + 2) * 4; }

// max_splits: the partials that the workspace holds (then nothing more is asked of it); total 0 if no size makes so few
dec_plan plan_decode(const kv_pool & p, int32_t n_seq, const int64_t * ctx, int32_t R, bool fine = true,
                     int64_t max_splits = kAnySplits) {
    dec_plan pl;
    const int32_t cus = device_cus(p.device());
    const split_choice pick = choose_split_stream(n_seq, ctx, p.h_kv(), cus, (R + 15) / 16, fine, max_splits);
    pl.split_tokens = pick.cells;
    int32_t asked = max_splits < kAnySplits ? pick.cells : pick.asked;
    // tuning knob for measurement: FNKV_SPLIT_TOKENS (a multiple of 32 from 256 to 4,096), read once per process
    static const int32_t split_knob = env_int_once("FNKV_SPLIT_TOKENS", 0);
    if (split_knob >= kPageTokens && split_knob <= kMaxSplitPages * kPageTokens && split_knob % kTileTokens == 0) {
        pl.split_tokens = asked = split_knob;
    }
    if (pl.split_tokens == 0) {
        return pl;
    }
    pl.split0[0] = 0;
    int64_t splits_asked = 0;
    for (int32_t i = 0; i < n_seq; ++i) {
        splits_asked += (ctx[i] + asked - 1) / asked;
        pl.split0[i + 1] = pl.split0[i] + static_cast<int32_t>((ctx[i] + pl.split_tokens - 1) / pl.split_tokens);
    }
    // one row tile (R <= 16): the splits of a sequence stride over its tiles, so at any moment the workgroups read
    // one window of the sequence together, and host and device contexts split alike (device contexts always stride:
    // decode_launch); more rows: contiguous splits
    pl.strided = R <= 16 ? 1 : 0;
    pl.total = pl.split0[n_seq];
    pl.fold_bytes = fold_region_bytes(p);
    pl.po_bytes = int64_t(pl.total) * p.h_kv() * R * kHeadDim * 4;
    pl.bytes = pl.fold_bytes + std::max<int64_t>(pl.total, splits_asked) * split_bytes(p, R);
    // the fold waits for the other splits of its pair, so every workgroup of the launch must be resident at once:
    // one a CU (the stream kernel's LDS)
    pl.fold = fold_enabled() && int64_t(pl.total) * p.h_kv() <= cus;
    return pl;
}

// The fold of at most kRowMergeSplits splits a row (every sparse launch's, most dense ones'): one workgroup a whole row
// (256 values), GRP waves = 64 float4 columns x GRP split groups (one a wave: group g folds splits g, g + GRP, ... with a
// running max, its loads in flight together), then the waves in order in LDS. An eighth of merge_kernel's workgroups: at
// these sizes a launch's cost is mostly the dispatch of its workgroups. The dense, the plain sparse and the gated form
// are instances of their own, so that a workgroup starts with only what its form needs: 8,192 rows of one split
// (16 sequences of 500-755 cells, T = 4, 128 heads on 16 KV heads) 23.4 us as one kernel for all forms, 19.6 as its own.
constexpr int32_t kRowMergeSplits = 96;
template <int GRP, bool SPARSE, bool GATED> __global__ __launch_bounds__(64 * GRP) void merge_row_kernel(merge_args a) {
    __shared__ float sM[GRP];
    __shared__ float sL[GRP];
    __shared__ floatx4 sA[GRP][64];
    const int32_t tid = static_cast<int32_t>(threadIdx.x);
    const int32_t c4 = tid & 63, g = tid >> 6;
    int32_t rest = static_cast<int32_t>(blockIdx.x);
    const int32_t r = rest % a.R;
    rest /= a.R;
    const int32_t kvh = rest % a.h_kv;
    const int32_t s = rest / a.h_kv;
    int32_t s0 = 0, n = 0;
    if (!merge_splits<SPARSE>(a, s, s0, n)) {
        return;
    }
    const int64_t row = (int64_t(s) * a.T + r / a.G) * a.hq + kvh * a.G + r % a.G;
    float4 gate = {};
    if (GATED && g == 0) { // requested beside the partials
        gate = finish_gate(a.fin, row, c4 * 4);
    }
    float m = kNegInf, l = 0.0f;
    int32_t bad = 0; // a split that saw an unmapped page marked its partial with a NaN max: nothing is written
    floatx4 A = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int32_t i = g; i < n; i += GRP) {
        const int64_t prow = (int64_t(s0 + i) * a.h_kv + kvh) * a.R + r;
        const float2 ml = *reinterpret_cast<const float2 *>(a.pml + prow * 2);
        bad |= ml.x != ml.x ? 1 : 0;
        const floatx4 o = *reinterpret_cast<const floatx4 *>(a.po + prow * kHeadDim + c4 * 4);
        const float m_new = fmaxf(m, ml.x);
        const float m_use = m_new == kNegInf ? 0.0f : m_new;
        const float f_old = __builtin_amdgcn_exp2f(m - m_use);
        const float f_new = __builtin_amdgcn_exp2f(ml.x - m_use);
        A = A * f_old + o * f_new;
        l = __builtin_fmaf(l, f_old, ml.y * f_new);
        m = m_new;
    }
    sA[g][c4] = A;
    if (c4 == 0) {
        sM[g] = m;
        sL[g] = l;
    }
    if (__syncthreads_or(bad)) {
        return;
    }
    if (g != 0) {
        return;
    }
    float Ms = sM[0], Ls = sL[0];
    floatx4 As = sA[0][c4];
#pragma unroll
    for (int32_t w = 1; w < GRP; ++w) {
        const float mn = fmaxf(Ms, sM[w]);
        const float mu = mn == kNegInf ? 0.0f : mn;
        const float f0 = __builtin_amdgcn_exp2f(Ms - mu), f1 = __builtin_amdgcn_exp2f(sM[w] - mu);
        As = As * f0 + sA[w][c4] * f1;
        Ls = __builtin_fmaf(Ls, f0, sL[w] * f1);
        Ms = mn;
    }
    if constexpr (GATED) {
        finish_gated(a.fin, row, c4 * 4, As, Ls, gate);
    } else {
        finish_plain(a.fin, row, c4 * 4, As, Ls);
    }
}

void launch_merge(const merge_args & m, hipStream_t st) {
    const dim3 rows(static_cast<uint32_t>(m.n_seq * m.h_kv * m.R));
    if (m.sel_splits > 0) { // a sparse launch (at most 17 splits a row)
        if (m.fin.gate != nullptr) {
            hipLaunchKernelGGL((merge_row_kernel<8, true, true>), rows, dim3(512), 0, st, m);
        } else {
            hipLaunchKernelGGL((merge_row_kernel<8, true, false>), rows, dim3(512), 0, st, m);
        }
        return;
    }
    // a workgroup a row up to 96 splits a sequence (67 splits fold faster so, 128 over more threads); otherwise a
    // workgroup a (row, 32 values)
    int32_t most = 0;
    for (int32_t i = 0; i < m.n_seq; ++i) {
        most = std::max(most, m.split0[i + 1] - m.split0[i]);
    }
    if (most <= kRowMergeSplits) {
        hipLaunchKernelGGL((merge_row_kernel<8, false, false>), rows, dim3(512), 0, st, m);
    } else {
        hipLaunchKernelGGL(merge_kernel, dim3(8 * rows.x), dim3(256), 0, st, m);
    }
}

} // namespace fnkv

using fnkv::set_error;

#ifdef FNKV_TIMING
static uint64_t * g_timing = nullptr;
extern "C" void fnkv_debug_timing(void * buf) { g_timing = static_cast<uint64_t *>(buf); }
namespace fnkv {
uint64_t * timing_buffer() { return g_timing; }
}
#endif

namespace fnkv {

// The dense decode launch: ctx holds each sequence's context (ctx_dev null) or the host's bound on the device word
// ctx_dev[i] (then the splits stride over the sequence's tiles, so every depth up to the bound spreads over the same
// grid, and a context outside T .. bound sets FNKV_DEV_ERR_DEPTH in *err and writes nothing for that sequence).
int decode_launch(const fnkv_pool * pool, int32_t n_seq, const int32_t * slots, const int64_t * ctx,
                  const int64_t * ctx_dev, uint32_t * err, int32_t T, int32_t layer, int32_t hq, float scale,
                  const void * q, const void * k_new, const void * v_new, int32_t new_dtype, void * out, void * ws,
                  int64_t ws_bytes, hipStream_t st, const char * who) {
    const std::string name(who);
    const kv_pool * p = pool_of(pool);
    if (p == nullptr || n_seq <= 0 || n_seq > FNKV_MAX_SEQS || slots == nullptr || ctx == nullptr || T <= 0 ||
        layer < 0 || layer >= p->layers() || hq <= 0 || hq % p->h_kv() != 0 || q == nullptr || out == nullptr ||
        ws == nullptr || !(scale > 0.0f) || !std::isfinite(scale) || ((k_new == nullptr) != (v_new == nullptr)) ||
        (new_dtype != FNKV_F16 && new_dtype != FNKV_F32)) {
        set_error(name + ": argument outside the contract");
        return FNKV_ERR_ARG;
    }
    const int32_t G = hq / p->h_kv();
    const int32_t R = G * T;
    if (R > FNKV_MAX_ROWS) {
        set_error(name + ": G * T = " + std::to_string(R) + " exceeds " + std::to_string(FNKV_MAX_ROWS));
        return FNKV_ERR_ARG;
    }
    if ((reinterpret_cast<uintptr_t>(q) & 15) != 0 || (reinterpret_cast<uintptr_t>(out) & 15) != 0 ||
        (reinterpret_cast<uintptr_t>(ws) & 15) != 0) {
        set_error(name + ": q, out and ws must be 16-byte aligned");
        return FNKV_ERR_ARG;
    }
    for (int32_t i = 0; i < n_seq; ++i) {
        if (slots[i] < 0 || slots[i] >= p->pages().n_slots() || ctx[i] < T || ctx[i] > p->mapped_cells(slots[i])) {
            set_error(name + ": sequence " + std::to_string(i) + " (slot " + std::to_string(slots[i]) + ", " +
                      (ctx_dev != nullptr ? "bound " : "ctx ") + std::to_string(ctx[i]) +
                      ") outside the slot's mapped cells");
            return FNKV_ERR_ARG;
        }
        // with the new cells written by the launch, two sequences in one slot would write the same cells
        for (int32_t k = 0; k < i && k_new != nullptr; ++k) {
            if (slots[k] == slots[i]) {
                set_error(name + ": slot " + std::to_string(slots[i]) + " appears twice in a launch that appends");
                return FNKV_ERR_ARG;
            }
        }
    }
    dec_plan pl = plan_decode(*p, n_seq, ctx, R);
    if (ws_bytes < pl.bytes) {
        // (a workspace sized for longer contexts can be smaller than the fine splits of short ones need)
        pl = plan_decode(*p, n_seq, ctx, R, false);
    }
    if (ws_bytes < pl.bytes) {
        // The rule's split count falls where the contexts outgrow one round of workgroups at one size and the next larger
        // size takes them in one (2 KV heads: 131,041 cells 128 splits, 140,000 cells 110), so a workspace sized for
        // deeper contexts can hold fewer splits than a shorter call's. It holds half a round's at least, and the deeper
        // call's size makes no more splits of the shorter contexts: the best of the sizes that it holds. (A workspace
        // below that and below the call's own stays refused.)
        const int64_t holds = (ws_bytes - fold_region_bytes(*p)) / split_bytes(*p, R);
        if (holds >= std::max(1, device_cus(p->device()) / (2 * p->h_kv()))) {
            const dec_plan held = plan_decode(*p, n_seq, ctx, R, false, holds);
            pl = held.total > 0 ? held : pl;
        }
    }
    if (ws_bytes < pl.bytes) {
        set_error(name + ": workspace too small");
        return FNKV_ERR_ARG;
    }
    dec_args a;
    a.pv = p->view();
    a.q = static_cast<const uint16_t *>(q);
    a.k_new = k_new;
    a.v_new = v_new;
    a.new_f32 = new_dtype == FNKV_F32 ? 1 : 0;
    a.po = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + pl.fold_bytes);
    a.pml = reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + pl.fold_bytes + pl.po_bytes);
    if (pl.fold) {
        a.fold = static_cast<uint32_t *>(ws);
        a.out = static_cast<uint16_t *>(out);
        a.fold_spin = fold_spin_ticks();
    }
    a.c2 = scale * 1.4426950408889634f;
    a.layer = layer;
    a.T = T;
    a.G = G;
    a.hq = hq;
    a.R = R;
    a.n_seq = n_seq;
    a.split_tokens = pl.split_tokens;
    a.strided = ctx_dev != nullptr ? 1 : pl.strided;
    a.ctx_dev = ctx_dev;
    a.err = err;
    for (int32_t i = 0; i < FNKV_MAX_SEQS; ++i) {
        a.slot[i] = i < n_seq ? slots[i] : 0;
        a.ctx[i] = i < n_seq ? ctx[i] : 0;
    }
    for (int32_t i = 0; i <= FNKV_MAX_SEQS; ++i) {
        a.split0[i] = i <= n_seq ? pl.split0[i] : pl.total;
    }
#ifdef FNKV_TIMING
    a.ts = g_timing;
#endif
    const dim3 grid(static_cast<uint32_t>(pl.total), static_cast<uint32_t>(p->h_kv()));
    launch_stream(p->device(), (R + 15) / 16, grid, a, st);
    if (pl.fold) {
        if (hipGetLastError() != hipSuccess) {
            set_error(name + ": launch failed");
            return FNKV_ERR_HIP;
        }
        return FNKV_OK;
    }
    merge_args m;
    m.po = a.po;
    m.pml = a.pml;
    m.fin.out = static_cast<uint16_t *>(out);
    m.T = T;
    m.G = G;
    m.hq = hq;
    m.R = R;
    m.h_kv = p->h_kv();
    m.n_seq = n_seq;
    m.ctx_dev = ctx_dev;
    m.T_dev = T;
    for (int32_t i = 0; i <= FNKV_MAX_SEQS; ++i) {
        m.split0[i] = a.split0[i];
    }
    for (int32_t i = 0; i < FNKV_MAX_SEQS; ++i) {
        m.cap[i] = a.ctx[i];
    }
    launch_merge(m, st);
    if (hipGetLastError() != hipSuccess) {
        set_error(name + ": launch failed");
        return FNKV_ERR_HIP;
    }
    return FNKV_OK;
}

// The no-allocation variant's workspace: the split partials of fnkv_attn_decode_noalloc live in this file-scope
// device array (each device that runs the library holds its own copy until the process ends). Host code never passes
// the array's name to a kernel (on the host it is only a stand-in for the symbol): it asks each device once, when the
// first pool on that device is created, for the array's device address and uses that.
//
// One device's array serves one (pool, stream) pair at a time: the first fnkv_attn_decode_noalloc call on a device
// binds it to that call's pool and stream, and calls from another pool or on another stream are refused (they could
// run while the bound pair's last call is still in flight) until the bound pool is destroyed, which drains the device
// and releases the binding.
constexpr int64_t kNoAllocScratchBytes = int64_t(16) << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

namespace {
constexpr int32_t kScratchDevices = 64;
struct scratch_binding {
    void * ptr = nullptr;               // the array's device address on this device
    const kv_pool * owner = nullptr;    // the pool bound to it, or null
    hipStream_t stream = nullptr;       // the stream its calls run on (valid while owner is set)
};
std::mutex g_scratch_mu;
scratch_binding g_scratch[kScratchDevices];
} // namespace

bool scratch_init(int32_t device, std::string & err) {
    if (device < 0 || device >= kScratchDevices) {
        err = "fnkv_pool_create: device index outside 0 .. 63";
        return false;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device].ptr != nullptr) {
        return true;
    }
    int32_t cur = 0;
    if (hipGetDevice(&cur) != hipSuccess || hipSetDevice(device) != hipSuccess) {
        err = "fnkv_pool_create: cannot make the pool's device current";
        return false;
    }
    void * ptr = nullptr;
    const hipError_t rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    (void)hipSetDevice(cur);
    if (rc != hipSuccess || ptr == nullptr) {
        err = std::string("fnkv_pool_create: hipGetSymbolAddress of the decode scratch failed: ") +
              hipGetErrorString(rc);
        return false;
    }
    g_scratch[device].ptr = ptr;
    return true;
}

void scratch_release(const kv_pool * pool) {
    const int32_t device = pool->device();
    if (device < 0 || device >= kScratchDevices) {
        return;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device].owner != pool) {
        return;
    }
    int32_t cur = 0;
    if (hipGetDevice(&cur) == hipSuccess && hipSetDevice(device) == hipSuccess) {
        (void)hipDeviceSynchronize();
        (void)hipSetDevice(cur);
    }
    g_scratch[device].owner = nullptr;
    g_scratch[device].stream = nullptr;
}

// the device address of the scratch for a call of `pool` on `stream`, binding the pair on the device's first call;
// null (with the error set) when another pool or stream holds it
static void * scratch_claim(const kv_pool * pool, hipStream_t stream) {
    const int32_t device = pool->device();
    if (device < 0 || device >= kScratchDevices) {
        set_error("fnkv_attn_decode_noalloc: device index outside 0 .. 63");
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    scratch_binding & b = g_scratch[device];
    if (b.ptr == nullptr) {
        set_error("fnkv_attn_decode_noalloc: the decode scratch of the pool's device was never looked up");
        return nullptr;
    }
    if (b.owner == nullptr) {
        b.owner = pool;
        b.stream = stream;
    } else if (b.owner != pool) {
        set_error("fnkv_attn_decode_noalloc: the device's scratch is bound to another pool (calls could overlap); "
                  "destroy that pool first or use fnkv_attn_decode_dev");
        return nullptr;
    } else if (b.stream != stream) {
        set_error("fnkv_attn_decode_noalloc: the device's scratch is bound to another stream of this pool (calls "
                  "could overlap); keep one stream or use fnkv_attn_decode_dev");
        return nullptr;
    }
    return b.ptr;
}

} // namespace fnkv

extern "C" {

int64_t fnkv_decode_workspace_bytes(const fnkv_pool * pool, int32_t n_seq, const int64_t * ctx, int32_t T, int32_t hq) {
    const fnkv::kv_pool * p = fnkv::pool_of(pool);
    if (p == nullptr || n_seq <= 0 || n_seq > FNKV_MAX_SEQS || ctx == nullptr || T <= 0 || hq <= 0 ||
        hq % p->h_kv() != 0) {
        return -1;
    }
    const int32_t R = (hq / p->h_kv()) * T;
    const fnkv::dec_plan pl = fnkv::plan_decode(*p, n_seq, ctx, R);
    return pl.bytes + 256;
}

void fnkv_test_decode_fold(int32_t mode, int64_t spin_ticks) {
    fnkv::g_fold_mode.store(mode < 0 ? -1 : (mode != 0 ? 1 : 0), std::memory_order_relaxed);
    fnkv::g_fold_spin.store(spin_ticks < 0 ? 20000 : spin_ticks, std::memory_order_relaxed);
}

int fnkv_attn_decode(const fnkv_pool * pool, int32_t n_seq, const int32_t * slots, const int64_t * ctx, int32_t T,
                     int32_t layer, int32_t hq, float scale, const void * q, const void * k_new, const void * v_new,
                     int32_t new_dtype, void * out, void * ws, int64_t ws_bytes, void * stream) {
    return fnkv::decode_launch(pool, n_seq, slots, ctx, nullptr, nullptr, T, layer, hq, scale, q, k_new, v_new,
                               new_dtype, out, ws, ws_bytes, static_cast<hipStream_t>(stream), "fnkv_attn_decode");
}

int fnkv_attn_decode_dev(const fnkv_pool * pool, int32_t n_seq, const int32_t * slots, const int64_t * ctx,
                         const int64_t * max_ctx, int32_t T, int32_t layer, int32_t hq, float scale, const void * q,
                         const void * k_new, const void * v_new, int32_t new_dtype, void * out, void * ws,
                         int64_t ws_bytes, uint32_t * err, void * stream) {
    if (ctx == nullptr || err == nullptr || (reinterpret_cast<uintptr_t>(ctx) & 7) != 0 ||
        (reinterpret_cast<uintptr_t>(err) & 3) != 0) {
        fnkv::set_error("fnkv_attn_decode_dev: ctx (8-byte aligned) and err (4-byte aligned) device words required");
        return FNKV_ERR_ARG;
    }
    return fnkv::decode_launch(pool, n_seq, slots, max_ctx, ctx, err, T, layer, hq, scale, q, k_new, v_new,
                               new_dtype, out, ws, ws_bytes, static_cast<hipStream_t>(stream),
                               "fnkv_attn_decode_dev");
}

int fnkv_attn_decode_noalloc(const fnkv_pool * pool, int32_t n_seq, const int32_t * slots, const int64_t * ctx,
                             const int64_t * max_ctx, int32_t T, int32_t layer, int32_t hq, float scale,
                             const void * q, const void * k_new, const void * v_new, int32_t new_dtype, void * out,
                             uint32_t * err, void * stream) {
    const fnkv::kv_pool * p = fnkv::pool_of(pool);
    if (p == nullptr || hq <= 0 || max_ctx == nullptr) {
        fnkv::set_error("fnkv_attn_decode_noalloc: argument outside the contract");
        return FNKV_ERR_ARG;
    }
    const int64_t need = fnkv_decode_workspace_bytes(pool, n_seq, max_ctx, T, hq);
    if (need < 0) {
        fnkv::set_error("fnkv_attn_decode_noalloc: argument outside the contract");
        return FNKV_ERR_ARG;
    }
    if (need > fnkv::kNoAllocScratchBytes) {
        fnkv::set_error("fnkv_attn_decode_noalloc: the launch needs " + std::to_string(need) +
                        " bytes of split partials, more than the library's fixed " +
                        std::to_string(fnkv::kNoAllocScratchBytes) + "-byte scratch (use fnkv_attn_decode_dev)");
        return FNKV_ERR_ARG;
    }
    if (ctx == nullptr || err == nullptr || (reinterpret_cast<uintptr_t>(ctx) & 7) != 0 ||
        (reinterpret_cast<uintptr_t>(err) & 3) != 0) {
        fnkv::set_error("fnkv_attn_decode_noalloc: ctx (8-byte aligned) and err (4-byte aligned) device words required");
        return FNKV_ERR_ARG;
    }
    void * ws = fnkv::scratch_claim(p, static_cast<hipStream_t>(stream));
    if (ws == nullptr) {
        return FNKV_ERR_ARG;
    }
    return fnkv::decode_launch(pool, n_seq, slots, max_ctx, ctx, err, T, layer, hq, scale, q, k_new, v_new, new_dtype,
                               out, ws, fnkv::kNoAllocScratchBytes, static_cast<hipStream_t>(stream),
                               "fnkv_attn_decode_noalloc");
}

} // extern "C"
